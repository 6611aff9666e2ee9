// Streaming skinny GEMM (decode path, M <= 16 typically) -- persistent, software-pipelined.
//
// Same math and epilogues as skinny_gemm.hip, restructured after rocprof showed the one-tile-
// per-workgroup kernel streaming weights at only ~3.1-3.4 TB/s: every workgroup paid launch +
// prologue + LDS reduction + epilogue around a single round trip of weight loads, leaving the
// CU's memory pipe idle between workgroups.  Here:
//
//  * X (the activation rows, <= ~140 KB) is staged in LDS once per workgroup and read back with
//    ds_read_b128 -- no activation loads in the weight stream, no X registers;
//  * the fused-RMSNorm row scales are computed once from that LDS copy;
//  * each workgroup is persistent over column tiles (tile = blockIdx.x + i*gridDim.x); its KS
//    waves split K, and every wave walks a flat list of (tile, k-batch) items;
//  * weight loads are raw buffer loads (SRD with num_records = N*K*2): the next item's 16 x
//    dwordx4 per lane are issued BEFORE the current item's MFMAs (two named register sets,
//    static indices -> counted vmcnt); k-groups that a wave does not have use an out-of-range offset
//    that the hardware answers with zeros and no memory traffic, but their addresses occupy its unit
//    as long as any load's: items past the last are not asked for, and a workgroup with one item takes
//    a form of as many k-groups as there are;
//  * the cross-wave reduction + fused epilogue of tile t runs while tile t+1's loads are in flight.
//
// XG variant (X does not fit in LDS: e.g. the down projection, K = 14336, with more than 5 rows):
// the activation fragments are streamed from global memory alongside the weights (X is a few
// hundred KB and stays L2-resident, so the extra loads hit L2, not HBM), with the same
// two-register-set pipeline; LDS holds an item of each wave and the reduction scratch.
#include "skinny_epilogue.h"

namespace {

// U: k-groups (128 wide) of an item, and ONE: every workgroup has one item, whose loads are all it asks for (launch()).
// Four waves: the registers that let as many workgroups share a CU as grid_of counts on.
template <int EPI, int NT, int KS, bool XG, int U, bool ONE>
__global__ __launch_bounds__(KS * 64, KS == 4 && EPI != EPI_QKV && !XG ? 3 : 1) void skinny_stream_kernel(
    SkinnyParams p, int nb, int tiles, int more, int xstride, int xskew) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int M = p.M, K = p.K, N = p.N;
  u16* xs = reinterpret_cast<u16*>(smem);
  // LDS-staged X: row m at m * xstride + (m / 4) * xskew elements.  xstride = K + 8 puts row m+1
  // one 16-B bank slot after row m; the extra 64-B skew every 4 rows (xskew 32) makes each
  // ds_read_b128 lane group ({0-3,12-15,20-27}, ...: rows nl, k-quarters g) hit 16 distinct slots
  // -- without it lanes (nl, g) and (nl + 4, g - 1)... share slots, a 2-way conflict on every read.
  const int xbytes = XG ? KS * U * 4096 : ((M * xstride * 2) + 4 * xskew * 2 + 15) & ~15;
  float* red = reinterpret_cast<float*>(smem + xbytes);  // [KS][NT][4][64]
  auto xrow = [&](int m) { return m * xstride + (m >> 2) * xskew; };
  float* rs = red + KS * NT * 4 * 64;                     // [16] row scales (1/rms, LayerNorm rstd)
  float* mu = rs + 16;                                    // [16] row means (folded LayerNorm)
  const float* mus = (p.fuse_rms == 2) ? mu : nullptr;
  const int lane = VWA_TX & 63, w = __builtin_amdgcn_readfirstlane(VWA_TX >> 6);
  const int nl = lane & 15, g = lane >> 4;

  EpiPre pre;
  epi_values<EPI, NT>(p, blockIdx.x, VWA_TX, pre);  // first tile's epilogue operands, early
  const int G = K / 128;
  const int gb = (G * w) / KS, ge = (G * (w + 1)) / KS;
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(p.W), (short)0, (int)((size_t)N * K * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(p.X), (short)0, (int)((size_t)M * p.ldx * 2), 0x00020000);
  const int my_tiles = ONE ? 1 : tiles + ((int)blockIdx.x < more);  // (of `tiles`, and the first `more` workgroups one more)
  // grammar-masked LM head (p.col_mask; the launcher keeps it only for NT 1, EPI store, LDS-staged
  // X and <= 64 tiles per workgroup): this workgroup's tiles that hold an admissible token of some
  // row, compacted into lanes (lane k: the k-th live tile).  Measured on the intent grammar: 42 %
  // of the LM head's tiles live per decode step on average, 10 % at the median.
  const bool masked = !ONE && NT == 1 && !XG && p.col_mask != nullptr;
  int n_live = my_tiles, live_tile = 0;
  if (masked) {
    const int tl = (int)blockIdx.x + lane * (int)gridDim.x;
    unsigned bits = 0;
    if (lane < my_tiles)
      for (int r = 0; r < p.col_mask_rows; ++r) bits |= p.col_mask[(size_t)r * p.col_mask_ld + (tl >> 1)];
    bits = (tl & 1) ? (bits >> 16) : (bits & 0xFFFFu);
    const unsigned long long live = __ballot(lane < my_tiles && bits != 0u);
    n_live = __popcll(live);
    const int rank = __popcll(live & ((1ull << lane) - 1ull));
    const int dst = ((live >> lane) & 1ull) ? rank : n_live + (lane - rank);  // a permutation of the lanes
    live_tile = __builtin_amdgcn_ds_permute(dst * 4, tl);
    if (n_live == 0) return;
  }
  // items: (tile t of this workgroup, k-batch b), one after another
  struct Item {
    int t, b;
  };
  auto next = [&](Item i) { return ++i.b == nb ? Item{i.t + 1, 0} : i; };
  auto tile_of = [&](Item i) { return masked ? __builtin_amdgcn_readlane(live_tile, i.t) : (int)blockIdx.x + i.t * (int)gridDim.x; };

  // Offsets: what the lanes differ in, and scalars (past the end: kOOB2, above every resource whatever is added).  One form for both
  // weight layouts, without branches: behind a join the compiler waits for as many loads as the shorter way in has.
  // XG: an item's X, 16 rows of U k-groups, is asked for 1 KB of rows at a time and turned to the fragments (lane (row nl, group g),
  // substep s: k 32 g + 8 s of the k-group) through the wave's own piece of LDS.  Asked for as fragments, a load touched 64 pieces of
  // 16 bytes 64 apart, four times the cycles of the address unit: 16 x 2048 x 8192 16.9 -> 11.9 us.  Chunk c of row r sits at slot
  // c ^ ((r + 4) & 15) of its 16: rows and chunks of a ds_read_b128's lane groups ({0-3,12-15,20-27}, ..) meet in no slot.
  constexpr int XC = 16 * U;  // 16-byte chunks of a row
  char* const xw = smem + w * (XG ? 16 * XC * 16 : 0);
  auto load_x = [&](uint4 (&xr)[U][4], Item i) {
    const int kg = gb + i.b * U;
#pragma unroll
    for (int j = 0; j < 4 * U; ++j) {
      const int row = (j * 64 + lane) / XC, c = (j * 64 + lane) % XC;
      const bool ok = i.t < n_live && row < M && kg + c / 16 < ge;
      xr[j / 4][j % 4] = bload_w_so<0>(rx, ok ? (unsigned)row * (unsigned)p.ldx * 2u + 16u * c : kOOB2, i.t < n_live ? kg * 256 : 0);
    }
  };
  auto turn_x = [&](const uint4 (&xr)[U][4]) {
#pragma unroll
    for (int j = 0; j < 4 * U; ++j) {
      const int row = (j * 64 + lane) / XC, c = (j * 64 + lane) % XC;
      *reinterpret_cast<uint4*>(xw + (row * XC + (c ^ ((row + 4) & 15))) * 16) = xr[j / 4][j % 4];
    }
    asm volatile("" ::: "memory");  // (a wave's LDS operations keep their order)
  };

  // pre-tiled: 1 KB contiguous per load instruction; row-major: 16 bytes of 64 pieces
  const unsigned w_lane = p.w_tiled ? lane * 16u : ((unsigned)nl * (unsigned)K + 32u * g) * 2u;
  const int w_kg = p.w_tiled ? 4096 : 256, w_s = p.w_tiled ? 1024 : 16;
  auto load_item = [&](uint4 (&wr)[NT][U][4], Item i) {
    const int tile = tile_of(i);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kg = gb + i.b * U + u;
      const bool ok = i.t < n_live && kg < ge;
      const unsigned voff = ok ? w_lane : kOOB2;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int at = ok ? (tile * NT + nt) * (32 * K) + kg * w_kg : 0;
#pragma unroll
        for (int s = 0; s < 4; ++s) wr[nt][u][s] = bload_w_so<0>(rw, voff, at + s * w_s);
      }
    }
  };

  f32x4 acc[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int xrl = xrow(min(nl, M - 1));  // (rows past the last: any values, no row of the results depends on another)
  auto compute_item = [&](const uint4 (&wr)[NT][U][4], const uint4 (&xr)[U][4], Item i) {
    if constexpr (XG) turn_x(xr);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kg = gb + i.b * U + u;
      if (kg >= ge) break;  // wave-uniform
      if constexpr (!ONE) __builtin_amdgcn_sched_barrier(0);  // (a k-group's fragments at a time: two items have the registers)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        uint4 a;
        if constexpr (XG) a = *reinterpret_cast<const uint4*>(xw + (nl * XC + 16 * u + ((4 * g + s) ^ ((nl + 4) & 15))) * 16);
        else a = *reinterpret_cast<const uint4*>(xs + xrl + kg * 128 + 32 * g + 8 * s);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = mfma16(as_bf16x8(a), as_bf16x8(wr[nt][u][s]), acc[nt]);
      }
    }
    if constexpr (XG) asm volatile("" ::: "memory");  // (the next item's rows take the place of these)
  };

  auto finish = [&](Item i) {  // behind a tile's last batch
    if (i.b == nb - 1)
      tile_epilogue<EPI, NT, KS, false>(p, red, rs, mus, tile_of(i), acc, w, lane, pre, !masked && i.t == 0);
  };

  uint4 A[NT][U][4], B[NT][U][4];
  uint4 XA[U][4], XB[U][4];  // XG only (dead otherwise)
  // ---- X rows into LDS, in batches of PB 16-byte pieces a thread whose loads are all on the way, the first batch in front of the
  // first weight item and the others behind it.  (Piece by piece each store waited for its own load and, vmcnt being in order, the
  // first one for the weights too: a chain of M K / 8 / threads round trips in front of any product.)
  constexpr int T = KS * 64, PB = KS == 4 ? 4 : 8;  // (four waves: three workgroups share a CU's registers)
  const int k8 = K / 8, pieces = M * k8;
  // (numbers of threads by a float reciprocal: small_div's bound)
  const float rk8 = __builtin_amdgcn_rcpf((float)k8);
  const int dm = (int)((T + 0.5f) * rk8), dk = T - dm * k8;
  int xm = (int)(((float)VWA_TX + 0.5f) * rk8), xk = VWA_TX - xm * k8;  // this thread's next piece
  u32x4 px[PB];
  auto walk = [&](int c0, auto&& f) {
    int m = xm, kk = xk;
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      if (c0 + i * T < pieces) f(i, m, kk);
      m += dm;
      kk += dk;
      if (kk >= k8) {
        kk -= k8;
        ++m;
      }
    }
    return make_int2(m, kk);
  };
  auto load_pieces = [&](int c0) {
    walk(c0, [&](int i, int m, int kk) {
      px[i] = gld(reinterpret_cast<const u32x4*>(p.X + (size_t)min(m, M - 1) * p.ldx + kk * 8));
    });
  };
  auto store_pieces = [&](int c0) {
    const int2 at = walk(c0, [&](int i, int m, int kk) {
      if (m < M) *reinterpret_cast<u32x4*>(xs + xrow(m) + kk * 8) = px[i];
    });
    xm = at.x;
    xk = at.y;
  };
  Item load{0, 0};
  if constexpr (!XG) load_pieces(0);
  load_item(A, load);
  if constexpr (XG) load_x(XA, load);
  if constexpr (!XG) {
    store_pieces(0);
    for (int c0 = PB * T; c0 < pieces; c0 += PB * T) {
      load_pieces(c0);
      store_pieces(c0);
    }
  }
  // the next item into a register set is issued right after that set's compute, BEFORE the tile
  // epilogue, so two items stay in flight through every epilogue
  auto load_next = [&](uint4 (&wr)[NT][U][4], uint4 (&xr)[U][4]) {
    load = next(load);
    load_item(wr, load);
    if constexpr (XG) load_x(xr, load);
  };
  if constexpr (!ONE) load_next(B, XB);
  if constexpr (!XG) lds_sync();
  // row scales (read behind the barrier of the first tile's reduction): rows w, w + KS, .. (two at a time where registers are free)
  constexpr int R = ONE ? 2 : 1;
  if (!p.fuse_rms) {
    if (VWA_TX < 16) rs[VWA_TX] = 1.f;
  } else {
    for (int m0 = w; m0 < M; m0 += R * KS) {
      float s[R] = {}, s1[R] = {};
      for (int k0 = lane; k0 < k8; k0 += 4 * 64) {
        uint4 v[R][4];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int kk = k0 + 64 * u, m = min(m0 + r * KS, M - 1);
            v[r][u] = make_uint4(0, 0, 0, 0);
            if (kk < k8)
              v[r][u] = XG ? *reinterpret_cast<const uint4*>(p.X + (size_t)m * p.ldx + kk * 8)
                           : *reinterpret_cast<const uint4*>(xs + xrow(m) + kk * 8);
          }
#pragma unroll
        for (int u = 0; u < 4; ++u)  // (pieces past the row's end add zeros)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            float f[8];
            unpack8(v[r][u], f);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              s[r] += f[j] * f[j];
              s1[r] += f[j];
            }
          }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        s[r] = wave_sum(s[r]);
        float sc, mean = 0.f;
        if (p.fuse_rms == 2) {  // LayerNorm: rstd from E[x^2] - mean^2
          mean = wave_sum(s1[r]) / (float)K;
          sc = rsqrtf(fmaxf(s[r] / (float)K - mean * mean, 0.f) + p.eps);
        } else {
          sc = rsqrtf(s[r] / (float)K + p.eps);
        }
        if (lane == 0 && m0 + r * KS < M) {
          rs[m0 + r * KS] = sc;
          mu[m0 + r * KS] = mean;
        }
      }
    }
  }

  if constexpr (ONE) {
    compute_item(A, XA, Item{0, 0});
    finish(Item{0, 0});
    return;
  }
  // The last items ask for nothing further: loads past the end bring no data, but their addresses take the unit as long as any
  const int n_items = n_live * nb;
  Item at{0, 0};
  int left = n_items;
  for (; left > 3; left -= 2) {
    compute_item(A, XA, at);
    load_next(A, XA);
    finish(at);
    at = next(at);
    compute_item(B, XB, at);
    load_next(B, XB);
    finish(at);
    at = next(at);
  }
  compute_item(A, XA, at);
  if (left == 3) load_next(A, XA);
  finish(at);
  if (left == 1) return;
  at = next(at);
  compute_item(B, XB, at);
  finish(at);
  if (left == 2) return;
  at = next(at);
  compute_item(A, XA, at);
  finish(at);
}

int g_x_skew = 32;  // LDS X row skew (elements per 4 rows; 0: none -- A/B knob, vwa_skinny_set_x_skew)

// Persistent workgroups of a launch: grid_cap (one a CU) times what a CU holds.  Of four waves (K < 2048; up to 188 registers) that
// is three, two of the QKV epilogue, where the X rows leave LDS for them: more weight bytes are on the way, and tiles past one a CU
// are not drawn one after the other.  us at one / two / three a CU, 8 rows: 5120 x 1280 10.7 / 9.9 / 9.9, 51872 x 1280 43.0 / 36.0 /
// 33.0, 32768 x 1024 27.5 / 21.9 / 21.0, 6144 x 1536 11.7 / 10.7 / 10.7; fp8 weights 32768 x 1024 17.5 / 15.8 / 14.8, 8192 x 1024 7.9 / 7.7
// / 7.6; up to 256 tiles the same launch.  (Measured before X was staged in batches and an fp8 row was quantised by one wave, which took
// 160 - 196 registers to 82 - 188: a CU holds as many workgroups as then.)
template <int EPI, int KS>
int grid_of(int ntiles, int grid_cap, size_t lds) {
  int per = KS == 4 ? EPI == EPI_QKV ? 2 : 3 : 1;
  while (per > 1 && per * lds > 160 * 1024) --per;
  return ntiles < grid_cap * per ? ntiles : grid_cap * per;
}

template <int EPI, int NT, int KS, bool XG, int U, bool ONE>
int launch_v(const SkinnyParams& p, hipStream_t st, int grid, size_t lds, int xstride, int nb) {
  const int ntiles = p.N / (16 * NT);
  hipLaunchKernelGGL((skinny_stream_kernel<EPI, NT, KS, XG, U, ONE>), dim3(grid), dim3(KS * 64), lds, st, p, nb, ntiles / grid,
                     ntiles % grid, xstride, XG ? 0 : g_x_skew);
  return 0;
}

template <int EPI, int NT, int KS>
int launch(const SkinnyParams& p0, hipStream_t st, int grid_cap) {
  SkinnyParams p = p0;
  const int xstride = p.K + 8;
  // (round 4's 17..64-row form -- X streamed next to the weights, 2 / 4 row fragments per weight
  // fragment -- measured slower than the tiled GEMM for whole decode steps and was removed in round
  // 5: more than 16 rows are the tiled GEMM's, gemm.hip)
  if (p.M > 16) return -10;
  const size_t xbytes = ((size_t)p.M * xstride * 2 + 4 * g_x_skew * 2 + 15) & ~(size_t)15;
  const size_t red = (size_t)(KS * NT * 4 * 64 + 32) * sizeof(float);  // + row scales + row means
  // X rows staged in LDS when they fit next to the reduction scratch; otherwise (the down
  // projection's 14336-wide rows at more than ~5 rows) streamed from L2 with the weights (XG)
  const bool lds_x = xbytes + red <= 160 * 1024;
  if (p.col_mask) {  // the masked tile list: NT 1, EPI store, LDS-staged X, <= 64 tiles per workgroup
    const int ntiles = p.N / (16 * NT), grid = grid_of<EPI, KS>(ntiles, grid_cap, xbytes + red);
    if (EPI != EPI_STORE || NT != 1 || !lds_x || (ntiles + grid - 1) / grid > 64 || p.col_mask_rows < 1)
      p.col_mask = nullptr;
  }
  constexpr int UX = 2 / NT;  // (XG)
  const size_t lds = lds_x ? xbytes + red : KS * UX * 4096 + red;
  const int ntiles = p.N / (16 * NT), grid = grid_of<EPI, KS>(ntiles, grid_cap, lds);
  const int per_wave = (p.K / 128 + KS - 1) / KS;  // k-groups of a tile's K that a wave has at most
  if (!lds_x) {
    if ((size_t)p.M * p.ldx * 2 >= 0x7FFFFFF0ull) return -10;
    return launch_v<EPI, NT, KS, true, UX, false>(p, st, grid, lds, xstride, (per_wave + UX - 1) / UX);
  }
  // One tile a workgroup whose k-groups a wave holds at once: the form without a second register set, of as many k-groups as there
  // are.  (The general one asked for two further items past the end and for the k-groups up to four that a wave does not have, each
  // as long in the address unit as a load that brings data.)  us in decoding, X staged piece by piece -> in batches -> with this form:
  // 16 x 2048 x 2048 9.2 -> 7.8 -> 4.9, 8 x 1280 x 1280 7.6 -> 6.5 -> 4.8, 8 x 5120 x 1280 with folded LayerNorm 10.1 -> 9.8 -> 7.2; general
  // form, its last items asking for none behind them: 16 x 16384 x 2048 (SwiGLU) 18.2 -> 15.7 -> 13.9.
  constexpr int U = 4 / NT;
  if (grid == ntiles && per_wave <= U && !p.col_mask) {
    if (per_wave <= 2) return launch_v<EPI, NT, KS, false, 2, true>(p, st, grid, lds, xstride, 1);
    if constexpr (U > 2) {
      if (per_wave == 3) return launch_v<EPI, NT, KS, false, 3, true>(p, st, grid, lds, xstride, 1);
      return launch_v<EPI, NT, KS, false, 4, true>(p, st, grid, lds, xstride, 1);
    }
  }
  return launch_v<EPI, NT, KS, false, U, false>(p, st, grid, lds, xstride, (per_wave + U - 1) / U);
}


// ------------------------------------------------------------------------------------------
// W8A8 variant (VWA_DTYPE=fp8): W is OCP e4m3 [N, K] bytes with per-row scales, X rows are
// quantised to e4m3 once per workgroup while staging into LDS (per-row dynamic scale
// amax/448), the inner product runs on the fp8 MFMA (16x16x32, 8 bytes per lane per operand),
// and both scales are applied in the epilogue.  Weight bytes per decode step are halved.
// ------------------------------------------------------------------------------------------
template <int EPI, int NT, int KS>
__global__ __launch_bounds__(KS * 64, KS == 4 && EPI != EPI_QKV ? 3 : 1) void skinny_fp8_kernel(SkinnyParams p, int nb, int xstride) {
  constexpr int U = 8 / NT;  // k-groups (128 wide) per item: 2 x b128 weight loads per k-group
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int M = p.M, K = p.K, N = p.N;
  uint8_t* xs = reinterpret_cast<uint8_t*>(smem);
  const int xbytes = ((M * xstride) + 15) & ~15;
  float* red = reinterpret_cast<float*>(smem + xbytes);  // [KS][NT][4][64]
  float* rs = red + KS * NT * 4 * 64;                     // [16] row scale (rms * x-quant scale)
  const int lane = VWA_TX & 63, w = __builtin_amdgcn_readfirstlane(VWA_TX >> 6);
  const int nl = lane & 15, g = lane >> 4;
  const int k8 = K / 8;

  EpiPre pre;
  epi_values<EPI, NT>(p, blockIdx.x, VWA_TX, pre);  // first tile's epilogue operands, early
  const int G = K / 128;
  const int gb = (G * w) / KS, ge = (G * (w + 1)) / KS;
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(p.W), (short)0, (int)((size_t)N * K), 0x00020000);
  const int ntiles = N / (16 * NT);
  const int my_tiles = (ntiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int n_items = my_tiles * nb;

  // (offsets as in skinny_stream_kernel.  fp8 tiled layout (ops.tile_weight_fp8): the (16-row tile, k-group) block is 2 KB
  // [s][lane][16 B], lane (nl, g) gets W[row][128 kg + 32 g + 16 s .. + 16), the same bytes as of row-major weights)
  const unsigned w_lane = p.w_tiled ? lane * 16u : (unsigned)nl * (unsigned)K + 32u * g;
  const int w_kg = p.w_tiled ? 2048 : 128, w_s = p.w_tiled ? 1024 : 16;
  auto load_item = [&](uint4 (&wr)[NT][U][2], int it) {
    const int tile = blockIdx.x + (it / nb) * gridDim.x;
    const int b = it % nb;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kg = gb + b * U + u;
      const bool ok = (it < n_items) && (kg < ge);
      const unsigned voff = ok ? w_lane : kOOB2;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int at = ok ? (tile * NT + nt) * (16 * K) + kg * w_kg : 0;
#pragma unroll
        for (int s = 0; s < 2; ++s) wr[nt][u][s] = bload_w_so<0>(rw, voff, at + s * w_s);
      }
    }
  };

  f32x4 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto compute_item = [&](const uint4 (&wr)[NT][U][2], int it) {
    const int b = it % nb;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kg = gb + b * U + u;
      if (kg >= ge) break;  // wave-uniform
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 a = make_uint4(0, 0, 0, 0);
        if (nl < M) a = *reinterpret_cast<const uint4*>(xs + nl * xstride + kg * 128 + 32 * g + 16 * s);
        const long a0 = (long)(((unsigned long)a.y << 32) | a.x), a1 = (long)(((unsigned long)a.w << 32) | a.z);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const uint4 v = wr[nt][u][s];
          const long b0 = (long)(((unsigned long)v.y << 32) | v.x), b1 = (long)(((unsigned long)v.w << 32) | v.z);
          acc[nt] = mfma16_fp8(a0, b0, acc[nt]);
          acc[nt] = mfma16_fp8(a1, b1, acc[nt]);
        }
      }
    }
  };

  uint4 A[NT][U][2], B[NT][U][2];
  // ---- rows w, w + KS, .. of X are this wave's: statistics (sum of squares for the fused RMSNorm, amax for the fp8 scale), then
  // e4m3 codes into LDS.  A row's first PB pieces a lane stay in registers in between, and the next row's are requested in front
  // of them, the first weight item behind the first row's.  (A row used to be read twice, one piece a lane waited for at a time, by its
  // own wave for the statistics and by all for the codes, and the weights were asked for behind both.  Not timed against that form; the
  // results are the same bits.)
  constexpr int PB = KS == 4 ? 4 : 8;  // (four waves: rows of less than 2048)
  u32x4 row[PB], ahead[PB];
  auto load_row = [&](u32x4 (&v)[PB], int m, int k0) {  // pieces past the row's end: zeros
#pragma unroll
    for (int u = 0; u < PB; ++u) {
      const int kk = k0 + 64 * u + lane;
      v[u] = u32x4{0, 0, 0, 0};
      if (m < M && kk < k8) v[u] = gld(reinterpret_cast<const u32x4*>(p.X + (size_t)m * p.ldx + kk * 8));
    }
  };
  load_row(ahead, w, 0);
  load_item(A, 0);
  for (int m = w; m < 16; m += KS) {
    float sc = 1.f;
    if (m < M) {
#pragma unroll
      for (int u = 0; u < PB; ++u) row[u] = ahead[u];
      load_row(ahead, m + KS, 0);
      float ss = 0.f, am = 0.f;
      for (int k0 = 0; k0 < k8; k0 += 64 * PB) {
        if (k0) load_row(row, m, k0);
#pragma unroll
        for (int u = 0; u < PB; ++u) {
          float f[8];
          unpack8(__builtin_bit_cast(uint4, row[u]), f);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            ss += f[j] * f[j];
            am = fmaxf(am, fabsf(f[j]));
          }
        }
      }
      ss = wave_sum(ss);
      am = wave_max(am);
      const float sx = am > 0.f ? am * (1.f / 448.f) : 1.f, iv = 1.f / sx;
      sc = (p.fuse_rms ? rsqrtf(ss / (float)K + p.eps) : 1.f) * sx;
      for (int k0 = 0; k0 < k8; k0 += 64 * PB) {
        if (k8 > 64 * PB) load_row(row, m, k0);
#pragma unroll
        for (int u = 0; u < PB; ++u) {
          const int kk = k0 + 64 * u + lane;
          float f[8];
          unpack8(__builtin_bit_cast(uint4, row[u]), f);
          uint2 q;
          q.x = cvt_pk_fp8(f[0] * iv, f[1] * iv) | (cvt_pk_fp8(f[2] * iv, f[3] * iv) << 16);
          q.y = cvt_pk_fp8(f[4] * iv, f[5] * iv) | (cvt_pk_fp8(f[6] * iv, f[7] * iv) << 16);
          if (kk < k8) *reinterpret_cast<uint2*>(xs + m * xstride + kk * 8) = q;
        }
      }
    }
    if (lane == 0) rs[m] = sc;
  }
  lds_sync();
  for (int it = 0; it < n_items; it += 2) {
    load_item(B, it + 1);
    compute_item(A, it);
    if (it % nb == nb - 1)
      tile_epilogue<EPI, NT, KS>(p, red, rs, nullptr, blockIdx.x + (it / nb) * gridDim.x, acc, w, lane, pre, it < nb);
    if (it + 1 >= n_items) break;
    load_item(A, it + 2);
    compute_item(B, it + 1);
    if ((it + 1) % nb == nb - 1)
      tile_epilogue<EPI, NT, KS>(p, red, rs, nullptr, blockIdx.x + ((it + 1) / nb) * gridDim.x, acc, w, lane, pre,
                                 it + 1 < nb);
  }
}

template <int EPI, int NT, int KS>
int launch_fp8(const SkinnyParams& p, hipStream_t st, int grid_cap) {
  constexpr int U = 8 / NT;
  // skinny_fp8_kernel holds 16 rows (rs[16], one MFMA row fragment): more rows must go to the
  // tiled GEMM, never to silently wrong rows 16+
  if (p.M > 16) return -10;
  const int G = p.K / 128;
  const int per_wave = (G + KS - 1) / KS;
  const int nb = (per_wave + U - 1) / U;
  const int xstride = p.K + 16;
  const size_t xbytes = ((size_t)p.M * xstride + 15) & ~(size_t)15;
  const size_t lds = xbytes + (size_t)(KS * NT * 4 * 64 + 32) * sizeof(float);
  if (lds > 160 * 1024) return -10;
  const int grid = grid_of<EPI, KS>(p.N / (16 * NT), grid_cap, lds);
  hipLaunchKernelGGL((skinny_fp8_kernel<EPI, NT, KS>), dim3(grid), dim3(KS * 64), lds, st, p, nb, xstride);
  return 0;
}

}  // namespace

// (round 4's 32-column tiles for the plain epilogues measured slower at
// 8 / 16 rows, profiles/r4_skinny_nt2_rows.jsonl, and were removed in round 5)

// Returns -10 when this shape does not fit the streaming kernel (caller falls back).
template <int KS>
int dispatch_ks(int epi, const SkinnyParams& p, int grid_cap, hipStream_t st) {
  if (p.w_scale) {
    switch (epi) {
      case EPI_STORE: return launch_fp8<EPI_STORE, 1, KS>(p, st, grid_cap);
      case EPI_RESID: return launch_fp8<EPI_RESID, 1, KS>(p, st, grid_cap);
      case EPI_GELU: return launch_fp8<EPI_GELU, 1, KS>(p, st, grid_cap);
      case EPI_SWIGLU: return launch_fp8<EPI_SWIGLU, 2, KS>(p, st, grid_cap);
      case EPI_QKV: return launch_fp8<EPI_QKV, 1, KS>(p, st, grid_cap);
      default: return -3;
    }
  }
  switch (epi) {
    case EPI_STORE: return launch<EPI_STORE, 1, KS>(p, st, grid_cap);
    case EPI_RESID: return launch<EPI_RESID, 1, KS>(p, st, grid_cap);
    case EPI_GELU: return launch<EPI_GELU, 1, KS>(p, st, grid_cap);
    case EPI_SWIGLU: return launch<EPI_SWIGLU, 2, KS>(p, st, grid_cap);
    case EPI_QKV: return launch<EPI_QKV, 1, KS>(p, st, grid_cap);
    case EPI_SPLIT: return p.n_q_heads % 16 || !p.q_out ? -4 : launch<EPI_SPLIT, 1, KS>(p, st, grid_cap);
    default: return -3;
  }
}

// Returns -10 when this shape does not fit the streaming kernel (caller falls back).
// ks = waves per workgroup splitting K (4 or 8); grid_cap = max persistent workgroups.
extern "C" void vwa_skinny_set_x_skew(int skew) { g_x_skew = skew == 0 ? 0 : 32; }

extern "C" int vwa_skinny_stream(int epi, const SkinnyParams* p, int grid_cap, int ks, hipStream_t st) {
  if (p->M < 1 || p->M > 16 || p->K % 128 != 0) return -10;
  if ((size_t)p->N * p->K * (p->w_scale ? 1 : 2) >= 0x7FFFFFF0ull) return -10;
  if (p->N < (epi == EPI_SWIGLU ? 32 : 16) || grid_cap < 1) return -2;  // (no tile: launch_v deals the tiles over the grid)
#ifdef VWA_ONLY_MULTI
  const int r = -10;
#else
  const int r = (ks == 4) ? dispatch_ks<4>(epi, *p, grid_cap, st) : dispatch_ks<8>(epi, *p, grid_cap, st);
#endif
  if (r) return r;
  return (int)hipGetLastError();
}
