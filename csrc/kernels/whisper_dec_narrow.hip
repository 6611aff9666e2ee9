// Persistent Whisper decoder step of narrow models (d = 128 .. 512, whisper-tiny and -base; ffn = 4 d, head_dim 64), one
// row: the whole token step in ONE launch like whisper_dec.hip, with THREE hand-offs between workgroups a layer instead of
// seven.  What bounds a narrow step is the number of dependent levels (one of whisper_dec.hip costs 4.1 us here whatever it computes:
// arrival, poll, the row's round trip, store drain; 33 of them are the 137 us of a whisper-tiny token, whose 68 MB take 11 us), so a
// workgroup that holds a slice of an activation multiplies it by its columns of the NEXT projection as well and hands on partial
// rows, which every consumer adds up in one order:
//   A  self     one workgroup per head: the layer's input row (sum of C's partials), LN1, the head's q / k / v columns,
//               cache write, self-attention, att_h . Wo[:, h]^T                                  -> H partial rows
//   B  cross    one per (head, quarter of the keys): x1 = x + sum of A's, LNx, the head's cross query, attention over its keys
//               (K / V in LDS by LDS-DMA a layer ahead), out . Wxo[:, h]^T                      -> 4 H partial rows and their
//               (max, sum), by which the consumers weigh them
//   C  ff       one per 64 hidden units: x2 = x1 + weighted sum of B's, LN2, GELU(fc1), f . W2[:, units]^T -> 4 H partial rows
// and the LM head on the remaining workgroups, whose vocabulary tiles are in registers before the last layer is done.
// d / 4 x 4 B partial rows of 6 (tiny) to 32 (base) producers are 9 - 64 KB a consumer: at d = 768 they would be 147 KB and
// cost what the hand-offs saved, so wider models keep whisper_dec.hip.
// Every role keeps its weights of the next layer in registers (<= 32 x 16 B a lane), refilled right after use.
// Same rounding as whisper_dec.hip (activations bf16, sums f32) but for two places, both finer: the cross query is one product
// of the normed row, and the cross-attention's output is not rounded at all (nd_attend: PIECES).
// Measured, whisper-tiny, 30 keys of context: 137 -> 62 us a token: 8.7 until the first layer's weights and keys are there (192 KB a
// head), A 4.6, B 4.5, C 3.6 a layer (tools/wdec_probe.py; the first layer's A 1.7 less: it waits for no rows), 4 for the LM head
// behind the last.  Of a phase the hand-off -- arrival to release -- is 0.5, a consumer's partial rows 1.0 - 1.4; the rest, 1.1 in C
// and 2.6 in A and B, are the phase's own products, attention and stores.
#include "whisper_dec.h"

namespace {
using namespace vwa;

enum { PH_A = 0, PH_B = 1, PH_C = 2 };  // level counters
constexpr int kChunks = 4;              // key chunks of a head (WdecParams::nch)
constexpr int kGenWord = 2048;          // (WdecParams::cnt u64 index: launches each workgroup completed)
constexpr int kLmTiles = 20;            // vocabulary tiles a workgroup has in flight
constexpr int L_PS = 1024;              // f32 [NG][D] partial sums of a row, <= 8 KB (behind the row, in front of L_RED)
constexpr int L_AV = L_VA + 512;        // bf16 [3][64] slice of an activation that meets the next projection: its pieces
constexpr int L_SK = 20480, L_SV = L_SK + 65536;  // self-attention: keys and values [512][64] bf16
static_assert(L_SV + 65536 <= kLds, "LDS");

template <int NS>
struct Nd {
  static constexpr int D = 128 * NS, H = 2 * NS, NT = D / 16;  // NT: column tiles of a D-wide projection
  static constexpr int NI = kChunks * H;                        // cross workgroups; ff workgroups (64 units each: 4 D / 64)
  static constexpr int C4 = D / 4, NG = kT / C4;                // a row by 4 columns a thread, NG groups of partial rows
  static constexpr int ROLES = H + 2 * NI;
  // WdecParams::part (f32): partial rows of A, B, C, B's (max, sum), the rows x, x1, x2 (bf16)
  static constexpr int PA = 0, PB = PA + H * D, PC = PB + NI * D, ML = PC + NI * D, ROWS = ML + 2 * NI, SIZE = ROWS + 3 * (D / 2);
  static_assert(NI * 64 == 4 * D && L_PS + NG * D * 4 <= L_RED, "roles; LDS");
};

VWA_DEVICE float bits_f(unsigned v) { return __uint_as_float(v); }

// (a kernel of its own stamps: 48 tests for null were 0.6 us of a token's 62)
template <bool TS>
VWA_DEVICE void nd_stamp(const WdecParams& p, int li, int phase, int k) {
  if constexpr (TS) wd_stamp(p, li, phase, k);
}

// the finished row (4 columns o of thread tx < C4) -> LDS, and to `keep`; returns (mean, 1 / std) to every thread
template <int NS>
VWA_DEVICE float2 nd_row(const WdecParams& p, const float (&o)[4], char* lds, u16* keep) {
  using N = Nd<NS>;
  constexpr int WV = (N::C4 + 63) / 64;  // waves that hold the row
  const int tx = VWA_TX;
  float* w8 = reinterpret_cast<float*>(lds + L_W8);
  if (tx < WV * 64) {
    float s = 0.f, s2 = 0.f;
    if (tx < N::C4) {
      u16 h[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        h[j] = f2bf(o[j]);
        const float f = bf2f(h[j]);
        s += f;
        s2 += f * f;
      }
      const u32x2 pk = {(unsigned)h[0] | ((unsigned)h[1] << 16), (unsigned)h[2] | ((unsigned)h[3] << 16)};
      *reinterpret_cast<u32x2*>(lds + L_XS + tx * 8) = pk;
      if (keep) __builtin_amdgcn_raw_buffer_store_b64(pk, rsrc_of(keep, N::D * 2), tx * 8, 0, 16);
    }
    s = wave_sum(s);
    s2 = wave_sum(s2);
    if ((tx & 63) == 0) {
      w8[tx >> 6] = s;
      w8[8 + (tx >> 6)] = s2;
    }
  }
  lds_sync();
  float s = w8[0], s2 = w8[8];
#pragma unroll
  for (int i = 1; i < WV; ++i) {
    s += w8[i];
    s2 += w8[8 + i];
  }
  constexpr float kInv = 1.f / N::D;
  const float mean = s * kInv;
  return make_float2(mean, rsqrtf(fmaxf(s2 * kInv - mean * mean, 0.f) + p.eps));
}

// the bias of thread tx's 4 columns, read ahead of the wait for the row
template <int NS>
VWA_DEVICE u32x2 nd_bias4(const u16* bias) {
  const int tx = VWA_TX;
  return bias && tx < Nd<NS>::C4 ? gld(reinterpret_cast<const u32x2*>(bias + 4 * tx)) : u32x2{0, 0};
}

// A phase's input row: base + bias + the sum of NP partial rows (MERGE: B's, item 4 h + c weighted by its share of head h's
// softmax sum), every load in flight at once, one order of the sum in every workgroup
template <int NS, int NP, bool MERGE>
VWA_DEVICE float2 nd_stage(const WdecParams& p, const float* part, const u16* base, u32x2 bb, char* lds, u16* keep) {
  using N = Nd<NS>;
  constexpr int R = (NP + N::NG - 1) / N::NG;
  constexpr unsigned kOut = 0x7FFFFFF0u;
  const int tx = VWA_TX, c = tx % N::C4, gi = tx / N::C4;
  float* ps = reinterpret_cast<float*>(lds + L_PS);
  const __amdgpu_buffer_rsrc_t rp = rsrc_of(part, (long long)NP * N::D * 4);
  float* cw = reinterpret_cast<float*>(lds + L_RED);
  u32x2 ml = {0, 0};
  if (MERGE && tx < NP) ml = __builtin_amdgcn_raw_buffer_load_b64(rsrc_of(p.part + N::ML, NP * 8), tx * 8, 0, 16);
  u32x4 v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = r * N::NG + gi;
    const bool in = gi < N::NG && i < NP;
    v[r] = __builtin_amdgcn_raw_buffer_load_b128(rp, (int)(in ? (unsigned)(i * N::D + 4 * c) * 4u : kOut), 0, 16);
  }
  u32x2 xb = {0, 0};
  if (tx < N::C4) xb = __builtin_amdgcn_raw_buffer_load_b64(rsrc_of(base, N::D * 2), c * 8, 0, 16);
  if constexpr (MERGE) {  // wave 0: every item's weight, a head's four side by side
    if (tx < 64) {
      const float l = bits_f(ml.y);
      float m = bits_f(ml.x);
      m = fmaxf(m, quad_xor<1>(m));
      m = fmaxf(m, quad_xor<2>(m));
      const float e = __expf(bits_f(ml.x) - m) * l;
      float den = e + quad_xor<1>(e);
      den += quad_xor<2>(den);
      if (tx < NP) cw[tx] = e / den;
    }
    lds_sync();
  }
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float w = MERGE ? cw[min(r * N::NG + gi, NP - 1)] : 1.f;  // (no such item: zeros were loaded)
    s[0] += w * bits_f(v[r].x);
    s[1] += w * bits_f(v[r].y);
    s[2] += w * bits_f(v[r].z);
    s[3] += w * bits_f(v[r].w);
  }
  if (gi < N::NG) *reinterpret_cast<float4*>(ps + gi * N::D + 4 * c) = make_float4(s[0], s[1], s[2], s[3]);
  lds_sync();
  float o[4] = {0.f, 0.f, 0.f, 0.f};
  if (tx < N::C4) {
#pragma unroll
    for (int g = 0; g < N::NG; ++g) {
      const float4 f = *reinterpret_cast<const float4*>(ps + g * N::D + 4 * tx);
      o[0] += f.x;
      o[1] += f.y;
      o[2] += f.z;
      o[3] += f.w;
    }
    const u16 x4[4] = {(u16)xb.x, (u16)(xb.x >> 16), (u16)xb.y, (u16)(xb.y >> 16)};
    const u16 b4[4] = {(u16)bb.x, (u16)(bb.x >> 16), (u16)bb.y, (u16)(bb.y >> 16)};
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (o[j] + bf2f(b4[j])) + bf2f(x4[j]);
  }
  return nd_row<NS>(p, o, lds, keep);
}

// the step's embedding row: from the tables (f32 sum of the two bf16 rows, one rounding), or x0; 4 columns of thread tx
template <int NS>
VWA_DEVICE void nd_embed(const WdecParams& p, float (&o)[4]) {
  using N = Nd<NS>;
  const int tx = VWA_TX;
  u32x2 a = {0, 0}, b = {0, 0};
  if (tx < N::C4) {
    if (p.tok_emb) {
      const int id = p.tokens[0], pos = p.positions[0];
      if (id >= 0 && id < p.emb_rows) a = gld(reinterpret_cast<const u32x2*>(p.tok_emb + (size_t)id * N::D + 4 * tx));
      b = gld(reinterpret_cast<const u32x2*>(p.pos_emb + (size_t)pos * N::D + 4 * tx));
    } else {
      a = gld(reinterpret_cast<const u32x2*>(p.x0 + 4 * tx));
    }
  }
  o[0] = bf2f((u16)a.x) + bf2f((u16)b.x);
  o[1] = bf2f((u16)(a.x >> 16)) + bf2f((u16)(b.x >> 16));
  o[2] = bf2f((u16)a.y) + bf2f((u16)b.y);
  o[3] = bf2f((u16)(a.y >> 16)) + bf2f((u16)(b.y >> 16));
}

// Weights of `tiles` 16-column tiles of a K = D projection: their 4 NS slices (of 32 k, 1 KB) each, dealt to the waves as one
// list, CNT a wave.  tile(j): the j-th tile's number.
template <int NS, int CNT, int O, int R, class F>
VWA_DEVICE void nd_load_tiles(const u16* W, int n_cols, uint4 (&wr)[R], F tile) {
  const __amdgpu_buffer_rsrc_t r = rsrc_of(W, (long long)n_cols * Nd<NS>::D * 2);
  const int tx = VWA_TX, lane = tx & 63, w = uni(tx >> 6);
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    const int u = w * CNT + i, j = u / (4 * NS), sl = u % (4 * NS);
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, (tile(j) * 4 * NS + sl) * 1024, 0);
    wr[O + i] = make_uint4(v.x, v.y, v.z, v.w);
  }
}
// half a tile: its slices 2 NS half .. + 2 NS (registers from O), one chain.  All 16 rows of A are the row -- a broadcast
// read, no lane waits for a branch -- and so are all rows of the result.
template <int NS, int O, int R>
VWA_DEVICE f32x4 nd_mma_half(const char* lds, const uint4 (&wr)[R], int half) {
  const u16* xs = reinterpret_cast<const u16*>(lds + L_XS) + 32 * ((VWA_TX & 63) >> 4);
  auto at = [](int sl) { return (sl >> 2) * 128 + 8 * (sl & 3); };
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2 * NS; ++i) {
    const uint4 a = *reinterpret_cast<const uint4*>(xs + (half ? at(2 * NS + i) : at(i)));
    acc = mfma16(as_bf16x8(a), as_bf16x8(wr[O + i]), acc);
  }
  return acc;
}

// Weights of all D output columns against 64 input values, k = 64 unit .. + 64 of a K = 128 KG projection: half of a k-group
// of the tiled layout (lane groups 2 hb, 2 hb + 1 of its four slices), two slices to a load: lane groups 0, 1 take slice 2 j,
// groups 2, 3 slice 2 j + 1.  Wave w: tiles w, w + 8, ..
template <int NS, int O, int R>
VWA_DEVICE void nd_load_k64(const u16* W, int KG, int unit, uint4 (&wr)[R]) {
  const __amdgpu_buffer_rsrc_t r = rsrc_of(W, (long long)Nd<NS>::D * KG * 256);
  const int tx = VWA_TX, lane = tx & 63, nl = lane & 15, g = lane >> 4, w = uni(tx >> 6);
  const int at = (g >> 1) * 1024 + (16 * (2 * (unit & 1) + (g & 1)) + nl) * 16;
#pragma unroll
  for (int t = 0; t < NS; ++t)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, at, ((w + 8 * t) * KG + (unit >> 1)) * 4096 + j * 2048, 0);
      wr[O + 2 * t + j] = make_uint4(v.x, v.y, v.z, v.w);
    }
}
// ... times the 64 values in LDS, each the sum of its PIECES, -> a partial row (piece i is row i of A: one product for all)
template <int NS, int O, int PIECES = 1, int R>
VWA_DEVICE void nd_k64(const char* lds, const uint4 (&wr)[R], float* out) {
  static_assert(PIECES <= 4, "rows of a lane");
  const int tx = VWA_TX, lane = tx & 63, g = lane >> 4, w = uni(tx >> 6);
  const u16* av = reinterpret_cast<const u16*>(lds + L_AV) + 64 * min(lane & 15, PIECES - 1);
  uint4 a[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) a[j] = *reinterpret_cast<const uint4*>(av + 32 * (g & 1) + 8 * (2 * j + (g >> 1)));
#pragma unroll
  for (int t = 0; t < NS; ++t) {
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; ++j) acc = mfma16(as_bf16x8(a[j]), as_bf16x8(wr[O + 2 * t + j]), acc);
    float v = acc[PIECES - 1];
#pragma unroll
    for (int e = PIECES - 2; e >= 0; --e) v += acc[e];  // (the small ones first)
    if (lane < 16) stf_sc1(out + (w + 8 * t) * 16 + lane, v);
  }
}

// four tiles of a K = D projection (the cross query of a head, 64 hidden units): column tx < 64, before bias and norm
template <int NS, int O, int R>
VWA_DEVICE float nd_cols64(char* lds, const uint4 (&wr)[R]) {
  float* red = reinterpret_cast<float*>(lds + L_RED);
  const int tx = VWA_TX, lane = tx & 63;
  const f32x4 acc = nd_mma_half<NS, O>(lds, wr, uni(tx >> 6) & 1);
  if (lane < 16) red[(tx >> 6) * 16 + lane] = acc[0];
  lds_sync();
  const int j = (tx & 63) >> 4, q = tx & 15;  // (two waves to a tile)
  return red[2 * j * 16 + q] + red[(2 * j + 1) * 16 + q];
}

VWA_DEVICE float nd_bias(const u16* b, int n) { return b ? bf2f(gld(b + n)) : 0.f; }

// Attention of the query in LDS (L_QF, bf16) over nk <= 512 keys in LDS, K rows at kl (16-byte piece c of key t at c ^ (t & 7)),
// V rows at vl; the normalized output goes to L_AV as bf16, or whole: PIECES 3 are its 24 bits in three bf16 numbers, so that what
// is not finished yet -- a quarter of a head's keys -- stays f32 through the matrix units too.  Logits of whisper-tiny against 64
// bits, mean of 8 utterances: whisper_dec.hip 5.67e-3, quarters rounded to one bf16 5.61e-3, this 5.55e-3 (and 0.3 us of a token's
// 62; 0.8 where each piece had a product of its own).
// Thread 0 gets (max, sum) of the scores' softmax.
// A wave takes tiles of 16 keys on its own -- max, weights, sum and output -- and one round puts the eight together:
//   scores: K as the MFMA's B operand, 16 keys to a tile, the wave's four tiles then one key a lane (products and sums as exact
//   as a chain of f32 FMAs: q and K are bf16);
//   values: 8 keys to a wave instruction, 16 bytes a lane, weights in f32; the lanes' sums halve what they hold at each step
// What bounds it is the instructions of a wave, two waves to a SIMD.  375 keys: a key per thread, 2 bytes of V a lane and three
// rounds of the workgroup 3.4 us, scores in every lane (four exponentials a tile) and full sums 2.0, this form 1.4.
template <int PIECES>
VWA_DEVICE float2 nd_attend(const WdecParams& p, int nk, const u16* kl, const u16* vl, char* lds) {
  static_assert(kT / 16 / 8 == 4, "a wave's tiles, one to a lane group");
  const int tx = VWA_TX, lane = tx & 63, nl = lane & 15, g = lane >> 4, w = uni(tx >> 6);
  float* P = reinterpret_cast<float*>(lds + L_P) + w * 64;  // this wave's weights
  float* ow = reinterpret_cast<float*>(lds + L_OW);
  float* w8 = reinterpret_cast<float*>(lds + L_W8);
  uint4 q[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) q[s] = *reinterpret_cast<const uint4*>(lds + L_QF + (32 * s + 8 * g) * 2);
  float sc = 0.f;
  const u16* kw = kl + (16 * w + nl) * 64;
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // tile w + 8 j
    if (16 * (w + 8 * j) >= nk) break;  // (uniform)
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s)
      acc = mfma16(as_bf16x8(q[s]), as_bf16x8(*reinterpret_cast<const uint4*>(kw + j * 8192 + (((4 * s + g) ^ (nl & 7)) << 3))), acc);
    sc = g == j ? acc[0] : sc;  // (key 16 (w + 8 j) + nl, in every row)
  }
  const bool valid = 16 * (w + 8 * g) + nl < nk;
  sc = valid ? sc * p.scale : -INFINITY;
  const float m = wave_max(sc);
  const float e = valid ? __expf(sc - m) : 0.f;
  P[lane] = e;
  const float l = wave_sum(e);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wave's own weights)
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int t0 = 16 * (w + 8 * (j >> 1)) + 8 * (j & 1);
    if (t0 >= nk) break;  // (uniform)
    const int t = min(t0 + (lane >> 3), nk - 1);  // (a key past the last: weight 0)
    const float pt = P[8 * j + (lane >> 3)];
    float f[8];
    unpack8(*reinterpret_cast<const uint4*>(vl + t * 64 + (lane & 7) * 8), f);
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] += pt * f[k];
  }
  // over the 8 keys of an instruction: lanes 32 apart (halves of the wave then hold dims 0-3 and 4-7 of the piece), 16 apart
  // (even and odd rows of 16: the first and last two of those), 8 apart
  auto swap_add = [](float a, float b, auto swap) {
    const auto r = swap(__float_as_uint(a), __float_as_uint(b));
    return bits_f(r[0]) + bits_f(r[1]);
  };
  auto by32 = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); };
  auto by16 = [](unsigned a, unsigned b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); };
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = swap_add(o[k], o[k + 4], by32);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    o[k] = swap_add(o[k], o[k + 2], by16);
    o[k] += row_ror<8>(o[k]);
  }
  if ((lane & 8) == 0)
    *reinterpret_cast<float2*>(ow + w * 64 + (lane & 7) * 8 + 4 * (lane >> 5) + 2 * ((lane >> 4) & 1)) = make_float2(o[0], o[1]);
  if (lane == 0) {
    w8[w] = m;
    w8[8 + w] = l;
  }
  lds_sync();
  float2 ml = make_float2(-INFINITY, 0.f);
  if (tx < 64) {
    float mw[8], lw[8], s = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      mw[k] = w8[k];
      lw[k] = w8[8 + k];
      ml.x = fmaxf(ml.x, mw[k]);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float e = __expf(mw[k] - ml.x);
      ml.y += e * lw[k];
      s += e * ow[k * 64 + tx];
    }
    float left = s / ml.y;
#pragma unroll
    for (int e = 0; e < PIECES; ++e) {
      const u16 b = f2bf(left);
      reinterpret_cast<u16*>(lds + L_AV)[64 * e + tx] = b;
      left = (b & 0x7F80) == 0x7F80 ? 0.f : left - bf2f(b);  // (infinities stay what they are)
    }
  }
  lds_sync();
  return ml;
}

// A: self-attention of head h and its part of the out-projection
template <int NS, bool TS>
VWA_DEVICE void nd_self(const WdecParams& p, int h, unsigned long long gen, char* lds) {
  using N = Nd<NS>;
  constexpr int NW = 8 * NS;
  uint4 wr[NW];
  const int NL = p.n_layers;
  auto load_qkv = [&](int li) {
    nd_load_tiles<NS, 6 * NS, 0>(p.layers[li].g[G_QKV].W, 3 * N::D, wr, [&](int j) { return (j >> 2) * N::NT + 4 * h + (j & 3); });
  };
  auto load_o = [&](int li) { nd_load_k64<NS, 6 * NS>(p.layers[li].g[G_O].W, NS, h, wr); };
  float x[4];
  nd_embed<NS>(p, x);
  load_qkv(0);
  const int ctx = min(p.ctx_lens[0], kT), bs = p.block_size;
  const long long slot = p.slots[0];
  long long old_at = 0;                   // this thread's key of the context (all but the newest), and the new one's row
  const bool old = VWA_TX < ctx - 1;
  if (old) old_at = (((long long)gld(p.block_table + p.seq_ids[0] * p.bt_stride + VWA_TX / bs) * p.H + h) * bs + VWA_TX % bs) * 64;
  const long long new_at = slot >= 0 ? ((slot / bs * p.H + h) * bs + slot % bs) * 64 : -1;
  load_o(0);
  u16* kl = reinterpret_cast<u16*>(lds + L_SK);
  u16* vl = reinterpret_cast<u16*>(lds + L_SV);
  u16* row = reinterpret_cast<u16*>(p.part + N::ROWS);
  for (int li = 0; li < NL; ++li) {
    const WdecLayer& L = p.layers[li];
    const int tx = VWA_TX, lane = tx & 63, w = tx >> 6;
    // ahead of the row: the context's keys and values (all but the newest), this thread's bias and LayerNorm column sum
    u32x4 kr[8], vr[8];
    if (old) {
      const u32x4* kp = reinterpret_cast<const u32x4*>(L.k_cache + old_at);
      const u32x4* vp = reinterpret_cast<const u32x4*>(L.v_cache + old_at);
#pragma unroll
      for (int c = 0; c < 8; ++c) kr[c] = gld(kp + c);
#pragma unroll
      for (int c = 0; c < 8; ++c) vr[c] = gld(vp + c);
    }
    float eb = 0.f, ec = 0.f;
    if (tx < 192) {
      const int n = ((tx >> 6) * N::NT + 4 * h + ((tx >> 4) & 3)) * 16 + (tx & 15);
      eb = nd_bias(L.g[G_QKV].bias, n);
      ec = gld(L.g[G_QKV].ln_c + n);
    }
    u16 *kc = L.k_cache, *vc = L.v_cache;
    const u32x2 bb = nd_bias4<NS>(li ? p.layers[li - 1].g[G_FC2].bias : nullptr);
    float2 st;
    u16* keep = h == 0 ? row : nullptr;
    nd_stamp<TS>(p, li, PH_A, 0);
    if (li == 0) {
      nd_stamp<TS>(p, li, PH_A, 1);
      st = nd_row<NS>(p, x, lds, keep);
    } else {
      wd_wait(p, PH_C, (gen * NL + li) * N::NI);
      nd_stamp<TS>(p, li, PH_A, 1);
      st = nd_stage<NS, N::NI, false>(p, p.part + N::PC, row + 2 * N::D, bb, lds, keep);
    }
    nd_stamp<TS>(p, li, PH_A, 2);
    // q, k, v of the head: 12 tiles over 8 waves -- one and a half a wave, three chains of half a tile
    float* red = reinterpret_cast<float*>(lds + L_RED);
    {
      const int odd = uni(w) & 1;
      const f32x4 a0 = nd_mma_half<NS, 0>(lds, wr, odd);
      const f32x4 am = nd_mma_half<NS, 2 * NS>(lds, wr, odd ^ 1);
      const f32x4 a1 = nd_mma_half<NS, 4 * NS>(lds, wr, odd);
      if (lane < 16) {
        red[w * 32 + lane] = a0[0] + ((w & 1) ? 0.f : am[0]);
        red[w * 32 + 16 + lane] = a1[0] + ((w & 1) ? am[0] : 0.f);
      }
    }
    if (old) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        *reinterpret_cast<u32x4*>(kl + tx * 64 + ((c ^ (tx & 7)) << 3)) = kr[c];
        *reinterpret_cast<u32x4*>(vl + tx * 64 + c * 8) = vr[c];
      }
    }
    lds_sync();
    if (tx < 192) {
      const int j = tx >> 4, q = tx & 15, r = j % 3, a = j / 3 * 64 + q;  // waves 2 (j / 3) and the next
      float v = r == 0 ? red[a] : r == 1 ? red[a + 16] + red[a + 32] : red[a + 48];
      v = (v - st.x * ec) * st.y + eb;
      const u16 o = f2bf(v);
      const int t4 = j & 3, dd = q < 8 ? 8 * t4 + q : 32 + 8 * t4 + q - 8, t = max(ctx - 1, 0);  // (ops.permute_qkv_rows)
      if (j < 4) reinterpret_cast<u16*>(lds + L_QF)[dd] = o;
      else if (j < 8) kl[t * 64 + (((dd >> 3) ^ (t & 7)) << 3) + (dd & 7)] = o;
      else vl[t * 64 + dd] = o;
      if (j >= 4 && new_at >= 0) *gp((j < 8 ? kc : vc) + new_at + dd) = o;
    }
    lds_sync();
    nd_attend<1>(p, ctx, kl, vl, lds);
    nd_k64<NS, 6 * NS>(lds, wr, p.part + N::PA + h * N::D);
    wd_arrive(p, PH_A);
    nd_stamp<TS>(p, li, PH_A, 3);
    if (li + 1 < NL) {
      load_qkv(li + 1);
      load_o(li + 1);
    }
  }
}

// B: cross-attention of (head, key chunk) and its part of the out-projection
template <int NS, bool TS>
VWA_DEVICE void nd_cross(const WdecParams& p, int item, unsigned long long gen, char* lds) {
  using N = Nd<NS>;
  constexpr int NW = 4 * NS;
  uint4 wr[NW];
  const int NL = p.n_layers, h = item / kChunks, nk = min(p.ch_len, p.T - item % kChunks * p.ch_len);
  auto load = [&](int li) {
    const WdecLayer& L = p.layers[li];
    nd_load_tiles<NS, 2 * NS, 0>(L.g[G_XQ].W, N::D, wr, [&](int j) { return 4 * h + j; });
    nd_load_k64<NS, 2 * NS>(L.g[G_XO].W, NS, h, wr);
    wd_kv_prefetch(p, li, item, lds);
  };
  load(0);
  u16* row = reinterpret_cast<u16*>(p.part + N::ROWS);
  for (int li = 0; li < NL; ++li) {
    const WdecLayer& L = p.layers[li];
    const int tx = VWA_TX;
    float eb = 0.f, ec = 0.f;
    if (tx < 64) {
      eb = nd_bias(L.g[G_XQ].bias, 64 * h + tx);
      ec = gld(L.g[G_XQ].ln_c + 64 * h + tx);
    }
    const u32x2 bb = nd_bias4<NS>(L.g[G_O].bias);
    nd_stamp<TS>(p, li, PH_B, 0);
    wd_wait(p, PH_A, (gen * NL + li + 1) * N::H);
    nd_stamp<TS>(p, li, PH_B, 1);
    const float2 st = nd_stage<NS, N::H, false>(p, p.part + N::PA, row, bb, lds, item == 0 ? row + N::D : nullptr);
    nd_stamp<TS>(p, li, PH_B, 2);
    const float v = nd_cols64<NS, 0>(lds, wr);
    if (tx < 64) reinterpret_cast<u16*>(lds + L_QF)[tx] = f2bf((v - st.x * ec) * st.y + eb);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share of the K / V chunk
    lds_sync();
    const float2 ml = nd_attend<3>(p, nk, reinterpret_cast<const u16*>(lds + L_KV), reinterpret_cast<const u16*>(lds + L_KV + L_KVV), lds);
    nd_k64<NS, 2 * NS, 3>(lds, wr, p.part + N::PB + item * N::D);
    if (tx == 0) {
      stf_sc1(p.part + N::ML + 2 * item, ml.x);
      stf_sc1(p.part + N::ML + 2 * item + 1, ml.y);
    }
    wd_arrive(p, PH_B);
    nd_stamp<TS>(p, li, PH_B, 3);
    if (li + 1 < NL) load(li + 1);
  }
}

// C: 64 hidden units of the feed-forward
template <int NS, bool TS>
VWA_DEVICE void nd_ff(const WdecParams& p, int unit, unsigned long long gen, char* lds) {
  using N = Nd<NS>;
  constexpr int NW = 4 * NS;
  uint4 wr[NW];
  const int NL = p.n_layers;
  auto load = [&](int li) {
    const WdecLayer& L = p.layers[li];
    nd_load_tiles<NS, 2 * NS, 0>(L.g[G_FC1].W, 4 * N::D, wr, [&](int j) { return 4 * unit + j; });
    nd_load_k64<NS, 2 * NS>(L.g[G_FC2].W, 4 * NS, unit, wr);
  };
  load(0);
  u16* row = reinterpret_cast<u16*>(p.part + N::ROWS);
  for (int li = 0; li < NL; ++li) {
    const WdecLayer& L = p.layers[li];
    const int tx = VWA_TX;
    float eb = 0.f, ec = 0.f;
    if (tx < 64) {
      eb = nd_bias(L.g[G_FC1].bias, 64 * unit + tx);
      ec = gld(L.g[G_FC1].ln_c + 64 * unit + tx);
    }
    const u32x2 bb = nd_bias4<NS>(L.g[G_XO].bias);
    nd_stamp<TS>(p, li, PH_C, 0);
    wd_wait(p, PH_B, (gen * NL + li + 1) * N::NI);
    nd_stamp<TS>(p, li, PH_C, 1);
    const float2 st = nd_stage<NS, N::NI, true>(p, p.part + N::PB, row + N::D, bb, lds, unit == 0 ? row + 2 * N::D : nullptr);
    nd_stamp<TS>(p, li, PH_C, 2);
    const float v = nd_cols64<NS, 0>(lds, wr);
    if (tx < 64) reinterpret_cast<u16*>(lds + L_AV)[tx] = f2bf(gelu_erf((v - st.x * ec) * st.y + eb));
    lds_sync();
    nd_k64<NS, 2 * NS>(lds, wr, p.part + N::PC + unit * N::D);
    wd_arrive(p, PH_C);
    nd_stamp<TS>(p, li, PH_C, 3);
    if (li + 1 < NL) load(li + 1);
  }
}

// greedy sample: the workgroup's best (every thread's bv / bi) -> its partial, arrival
VWA_DEVICE void nd_sample_part(const WdecParams& p, int m, char* lds, float bv, int bi) {
  const int tx = VWA_TX;
  float* w8 = reinterpret_cast<float*>(lds + L_W8);
#pragma unroll
  for (int k = 32; k > 0; k >>= 1) {
    const float ov = __shfl_xor(bv, k, 64);
    const int oi = __shfl_xor(bi, k, 64);
    argmax_merge(bv, bi, ov, oi);
  }
  lds_sync();
  if ((tx & 63) == 0) {
    w8[tx >> 6] = bv;
    w8[8 + (tx >> 6)] = __int_as_float(bi);
  }
  lds_sync();
  if (tx == 0) {
    for (int k = 1; k < 8; ++k) argmax_merge(bv, bi, w8[k], __float_as_int(w8[8 + k]));
    stf_sc1(p.smp_part + 2 * m, bv);
    stf_sc1(p.smp_part + 2 * m + 1, __int_as_float(bi));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_fetch_add(gp(p.cnt + kSmpCnt + 16 * (m & 7)), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// workgroup 0, behind its last layer: merge the n partials, advance the device loop
VWA_DEVICE void nd_sample_merge(const WdecParams& p, int n, unsigned long long base) {
  const int tx = VWA_TX;
  if (tx >= 64) return;
  int spins = 0;
  while ((long long)(cnt_sum8(p.cnt + kSmpCnt) - (base + (unsigned long long)n)) < 0) {
    __builtin_amdgcn_s_sleep(1);
    if (++spins > kSpinLimit) {
      if (tx == 0) set_err(p);
      break;
    }
  }
  float v = -INFINITY;
  int ix = 0x7fffffff;
  for (int k = tx; k < n; k += 64) argmax_merge(v, ix, ldf_sc1(p.smp_part + 2 * k), __float_as_int(ldf_sc1(p.smp_part + 2 * k + 1)));
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) {
    const float ov = __shfl_xor(v, m, 64);
    const int oi = __shfl_xor(ix, m, 64);
    argmax_merge(v, ix, ov, oi);
  }
  if (tx == 0) wd_advance(p, v == -INFINITY ? -1 : ix);
}

// LM head on the workgroups without a role (m of n): tiles m, m + n, ..; kLmTiles of them in registers ahead of the last row
template <int NS>
VWA_DEVICE void nd_head(const WdecParams& p, int m, int n, unsigned long long gen, char* lds) {
  using N = Nd<NS>;
  constexpr int SL = (4 * NS + 7) / 8;  // slices of a tile and wave
  uint4 wr[kLmTiles][SL];
  const int NV = p.n_vocab >> 4, mine = m < NV ? (NV - 1 - m) / n + 1 : 0;
  const int tx = VWA_TX, lane = tx & 63, g = lane >> 4, w = uni(tx >> 6);
  const __amdgpu_buffer_rsrc_t r = rsrc_of(p.lm_W, (long long)p.n_vocab * N::D * 2);
  float lc = 0.f, lb = 0.f;  // (thread t < 16 kLmTiles: column t & 15 of slot t / 16)
  bool mk = false;
  auto load = [&](int j0) {
#pragma unroll
    for (int s = 0; s < kLmTiles; ++s)
#pragma unroll
      for (int i = 0; i < SL; ++i) {
        const bool in = j0 + s < mine && w + 8 * i < 4 * NS;
        const int t = m + (j0 + s) * n;
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, in ? lane * 16 : 0x7FFFFFF0, in ? (t * 4 * NS + w + 8 * i) * 1024 : 0, 0);
        wr[s][i] = make_uint4(v.x, v.y, v.z, v.w);
      }
    const int col = (m + (j0 + (tx >> 4)) * n) * 16 + (tx & 15);
    if (tx < 16 * kLmTiles && j0 + (tx >> 4) < mine) {
      lc = gld(p.lm_c + col);
      lb = nd_bias(p.lm_b, col);
      mk = p.smp_mask && ((gld(p.smp_mask + (col >> 5)) >> (col & 31)) & 1u);
    }
  };
  load(0);
  const u32x2 bb = nd_bias4<NS>(p.layers[p.n_layers - 1].g[G_FC2].bias);
  // (polled seldom until the last layer's feed-forward arrives: the line is the one its workgroups add to)
  if (tx < 64) {
    const unsigned long long want = (gen + 1) * p.n_layers * N::NI;
    int spins = 0;
    while (true) {
      const long long left = (long long)(want - cnt_sum8(lvl_cnt(p, PH_C)));
      if (left <= 0) break;
      if (left > N::NI) __builtin_amdgcn_s_sleep(64);
      else __builtin_amdgcn_s_sleep(2);
      if ((spins & 255) == 255 && __hip_atomic_load(gp(p.cnt + kErrWord), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
      if (++spins > kSpinLimit) {
        if (tx == 0) set_err(p);
        break;
      }
    }
  }
  lds_sync();
  const u16* row = reinterpret_cast<const u16*>(p.part + N::ROWS);
  const float2 st = nd_stage<NS, N::NI, false>(p, p.part + N::PC, row + 2 * N::D, bb, lds, nullptr);
  const u16* xs = reinterpret_cast<const u16*>(lds + L_XS);
  float* red = reinterpret_cast<float*>(lds + L_KV);  // [8][kLmTiles][16]
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int j0 = 0; j0 < mine; j0 += kLmTiles) {
    uint4 a[SL];
#pragma unroll
    for (int i = 0; i < SL; ++i) {
      const int sl = w + 8 * i;
      a[i] = make_uint4(0, 0, 0, 0);
      if (sl < 4 * NS) a[i] = *reinterpret_cast<const uint4*>(xs + (sl >> 2) * 128 + 32 * g + 8 * (sl & 3));
    }
#pragma unroll
    for (int s = 0; s < kLmTiles; ++s) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < SL; ++i) acc = mfma16(as_bf16x8(a[i]), as_bf16x8(wr[s][i]), acc);
      if (lane < 16) red[(w * kLmTiles + s) * 16 + lane] = acc[0];
    }
    lds_sync();
    if (tx < 16 * kLmTiles && j0 + (tx >> 4) < mine) {
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) v += red[k * kLmTiles * 16 + tx];
      const int col = (m + (j0 + (tx >> 4)) * n) * 16 + (tx & 15);
      const float lg = (v - st.x * lc) * st.y + lb;
      *gp(p.logits + col) = lg;
      if (mk) argmax_merge(bv, bi, lg, col);
    }
    lds_sync();  // (red is rewritten)
    if (j0 + kLmTiles < mine) load(j0 + kLmTiles);
  }
  if (p.smp_mask) nd_sample_part(p, m, lds, bv, bi);
}

template <int NS, bool TS>
__global__ __launch_bounds__(kT) void wdec_narrow_kernel(WdecParams p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  using N = Nd<NS>;
  const int b = blockIdx.x, n = (int)gridDim.x - N::ROLES;
  // launches this workgroup completed = completed launches: the base of every level counter, whenever a workgroup starts
  const unsigned long long g0 = __hip_atomic_load(gp(p.cnt + kGenWord + b), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long gen = __builtin_amdgcn_readfirstlane((unsigned)g0) |
                                 ((unsigned long long)__builtin_amdgcn_readfirstlane((unsigned)(g0 >> 32)) << 32);
  // (the sampler's arrivals need every level, and so this read)
  const unsigned long long smp = p.smp_mask && b == 0 && VWA_TX < 64 ? cnt_sum8(p.cnt + kSmpCnt) : 0;
  if (b < N::H) nd_self<NS, TS>(p, b, gen, lds);
  else if (b < N::H + N::NI) nd_cross<NS, TS>(p, b - N::H, gen, lds);
  else if (b < N::ROLES) nd_ff<NS, TS>(p, b - N::H - N::NI, gen, lds);
  else if (p.lm_W) nd_head<NS>(p, b - N::ROLES, n, gen, lds);
  if (p.smp_mask && b == 0) nd_sample_merge(p, n, smp);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (VWA_TX == 0) __hip_atomic_store(gp(p.cnt + kGenWord + b), gen + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int NS>
int nd_launch(const WdecParams& p, int grid, hipStream_t st) {
  if (grid < Nd<NS>::ROLES + 16) return -10;
  if (p.ts) hipLaunchKernelGGL((wdec_narrow_kernel<NS, true>), dim3(grid), dim3(kT), kLds, st, p);
  else hipLaunchKernelGGL((wdec_narrow_kernel<NS, false>), dim3(grid), dim3(kT), kLds, st, p);
  return (int)hipGetLastError();
}

}  // namespace

// f32 numbers of WdecParams::part, 0: a model this kernel does not take
extern "C" int64_t vwa_wdec_narrow_part(int d) {
  switch (d) {
    case 128: return Nd<1>::SIZE;
    case 256: return Nd<2>::SIZE;
    case 384: return Nd<3>::SIZE;
    case 512: return Nd<4>::SIZE;
    default: return 0;
  }
}

extern "C" int vwa_wdec_narrow_launch(const WdecParams* p, int grid, hipStream_t st) {
  if (p->ffn != 4 * p->d || p->H * 64 != p->d || p->n_layers < 1 || p->nch != kChunks || p->ch_len > kMaxChunk ||
      p->ch_len * kChunks < p->T || p->ch_len * (kChunks - 1) >= p->T || !p->part || !p->lm_W)
    return -10;
  switch (p->d) {
    case 128: return nd_launch<1>(*p, grid, st);
    case 256: return nd_launch<2>(*p, grid, st);
    case 384: return nd_launch<3>(*p, grid, st);
    case 512: return nd_launch<4>(*p, grid, st);
    default: return -10;
  }
}
