// LDS-tiled MFMA GEMM for what the skinny decode kernels do not take (K12): the prompt suffix prefill of the intent
// LLM (apps/brain/src/server.ts:98-105: ~1.1k-token prompt, the un-cached suffix), continuous-batching steps of
// 17..64 rows, the Whisper encoder (1500 rows per utterance), and fewer rows of large pre-tiled bf16 weights
// (ops.rows_take_tiles).  Replaces hipBLASLt for every projection of both models.
//
//   Y[M, N] = epi( rstd[m] * (X[M, K] . W[N, K]^T) )       X bf16 row-major, f32 accumulate
//
// W layouts:
//   * tiled (ops.tile_weight, the decode kernels' layout -- the model keeps ONE copy of each
//     weight): per 16-row tile T and 128-wide k-group kg a contiguous 4 KB block
//     [s 0..3][lane 0..63][8] with lane = 16 g + n holding W[16 T + n][128 kg + 32 g + 8 s + e],
//     i.e. exactly the MFMA B fragments: the block is copied to LDS verbatim;
//   * row-major [N, K] (Whisper weights, tests): each 16-byte piece is scattered into the same
//     fragment-ordered LDS image while staging.
// Which k of a k-group a stage takes, and in which order, follows from the X rows' cache lines (swzk, gemm_stage.h).
//
// Tiling (gfx950, wave64), 128 x 128: workgroup = 4 waves (2 x 2), half a k-group (64 deep) per stage: A [128 rows][64
// k] (16 KB, chunk-XOR swizzled: conflict-free ds_read_b128) and B [8 tiles][2 MFMAs][64 lanes][8] (16 KB, fragment
// order -> every ds_read_b128 is 1 KB contiguous).  Each wave owns 64 x 64 = 4 x 4 MFMA tiles
// (mfma_f32_16x16x32_bf16, 32 MFMAs per stage).  Two stages in LDS (64 KB -> 2 workgroups per CU), filled by LDS-DMA one
// stage ahead.  256 x 256 (CfgP8): below.
// Grid: (row blocks x column blocks) remapped XCD-aware so the row blocks of one column block
// (same weight tile) share an XCD's L2, x split-K slices when the tile count alone cannot
// fill the 256 CUs (weight-streaming shapes: few rows) -- slices write f32 partials, a second
// kernel sums them and applies the epilogue.
//
// Epilogues (fused, after the optional per-row RMSNorm scale rstd -- gammas are folded into W):
//   0 store (+bias; bf16 or f32 out)   1 residual add (+bias)   2 SwiGLU over gate/up tiles
//   interleaved per 16 rows (ops.interleave_gate_up)   3 GELU (+bias)   4 GELU (+bias) then a
//   residual add (the Whisper conv stem's positional embedding: y = gelu(conv + b) + pos)
//   5 QKV (rotary + paged KV write)   6 split: the first n_split columns stored, relu^2 of the others
//   to a second matrix (one projection feeding a layer's mixers and its feed-forward)
//
// Grouped launches (routed experts, GemmParams::g_*): a row block is a tile of (row, expert) pairs of one
// expert; its X rows are gathered (or taken in place order) by the LDS-DMA's per-lane addresses, W is the
// expert's, and the per-row scale is the pair's score.
//
// Implicit-GEMM convolution (K3, ops.conv1d_gelu): X rows are ldx apart and K long, so a k=3
// conv over a zero-padded channels-last buffer is X row t = padded rows t*stride .. t*stride+2
// (ldx = stride*Cin, K = 3*Cin) -- the A tiles are staged through the same LDS-DMA pipeline.
#include "common.h"
#include "gemm_stage.h"
#include "vwa_kernels.h"

using namespace vwa;

namespace {

enum Epi { EPI_STORE = 0, EPI_RESID = 1, EPI_SWIGLU = 2, EPI_GELU = 3, EPI_GELU_RESID = 4, EPI_QKV = 5, EPI_SPLIT = 6 };
template <int EPI> constexpr bool kResid = EPI == EPI_RESID || EPI == EPI_GELU_RESID;
template <int EPI> constexpr bool kGelu = EPI == EPI_GELU || EPI == EPI_GELU_RESID;

constexpr int BKG = 128;
constexpr int kGroup = 4;  // row blocks of a grouped launch that walk the columns together

// Workgroup shapes: BM x BN output tile, WM x WN waves, each wave (BM/WM) x (BN/WN).
//   CfgS, 128 x 128: 4 waves of 64 x 64, 64 KB LDS, two workgroups per CU: few or odd tiles
//   CfgP8, 256 x 256: 8 waves of 128 x 64, 144 KB, one per CU: a quarter less read from LDS per MFMA where its tiles fill the
//     CUs (1011 x 28672 x 4096 237 -> 179 us) or their slices do (choose())
//   CfgF, CfgFs: <= 64 and <= 32 rows, bf16 or fp8 weights
// GROUPS: groups of WM x WN waves that take the stages of K in turn; their sums are added in LDS
template <int BM_, int BN_, int WM_, int WN_, int GROUPS_ = 1>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, GROUPS = GROUPS_, NW = WM_ * WN_, THREADS = 64 * NW * GROUPS;
  static constexpr int FM = BM / WM / 16, FN = BN / WN / 16;  // MFMA fragments per wave
  static constexpr int A_BYTES = BM * 128, STAGE = BM * 128 + BN * 128;
  // W8A16 stage: a full k-group -- two bf16 A half images + the fp8 B block of every tile
  static constexpr int W8STAGE = 2 * BM * 128 + BN * 128;
  static constexpr int NCOL_MAX = BN / WN;
  static constexpr int EPI_LDS = NW * (FM * 16) * (NCOL_MAX * 2 + 16);
  static constexpr int NST = BM <= 32 ? 4 : BM <= 64 ? 3 : 2;   // stage buffers: few rows take what lets two workgroups share a CU
  static constexpr int LDS = GROUPS * NST * STAGE > EPI_LDS ? GROUPS * NST * STAGE : EPI_LDS;
  static constexpr int W8NST = BM <= 32 ? 3 : 2;
  static constexpr int W8LDS = W8NST * W8STAGE > EPI_LDS ? W8NST * W8STAGE : EPI_LDS;
  static_assert((BM / 8) % NW == 0 && (BN / 8) % NW == 0, "whole LDS-DMA instructions per wave");
};
using CfgS = Cfg<128, 128, 2, 2>;
// The same with two groups of four waves that take the stages in turn, one workgroup per CU: below.
using CfgK = Cfg<128, 128, 2, 2, 2>;
using CfgKw = Cfg<128, 192, 2, 2, 2>;
// Few rows (<= 64: one row block): 64 x 128, 4 waves of 64 x 32, 2 workgroups per CU.  Such a product is weights arriving and
// little else, so what counts is how many of their bytes are on the way.
// bf16: three 24 KB stages where the 128-row tile had two of 32 KB, half of them rows that are not there (and one stage in flight
// behind the one being read).  32 rows: 28672 x 4096 53.7 -> 44.9 us, 6144 x 4096 19.4 -> 16.6; 48 rows: 4096 x 4096 15.7 -> 14.2.
// W8A16: 32 KB stages (16 KB of fp8 weights each -- the W8A8 kernel's weight bytes per stage: a half-k-group bf16-style stage
// carried 8 KB and measured 1.25x slower whole decode steps)
using CfgF = Cfg<64, 128, 1, 4>;
// ... of <= 32 rows: bf16 four stages of 20 KB; fp8 24 KB stages, so three fit where two did and two are in flight behind the one
// being read (32 rows: 28672 x 4096 23.3 us, 4096 x 4096 10.1 and 4096 x 14336 17.6 in eight slices with their sum; six stages here and
// four of 64 rows, one workgroup to a CU: 24.3, 10.7, 19.1, and 3 - 15 % slower over 21 weights)
using CfgFs = Cfg<32, 128, 1, 4>;
// ... of few columns as well: 64 columns to a tile, so that twice the CUs draw weights (narrow())
using CfgN = Cfg<64, 64, 1, 4>;
using CfgNs = Cfg<32, 64, 1, 4>;

// buffer resource over [base, base + bytes): loads past the end return zero (rows >= M, weight
// tiles >= N), so the stage issue needs no bounds branches
VWA_DEVICE __amdgpu_buffer_rsrc_t rsrc(const void* base, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0,
                                           (int)(bytes < 0x7FFFFFF0ull ? bytes : 0x7FFFFFF0ull), 0x00020000);
}

VWA_DEVICE void dma16(__amdgpu_buffer_rsrc_t r, char* lds_wave_base, unsigned voff, unsigned soff = 0) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds_wave_base, 16, voff, soff, 0,
                                           0);
}

// Stage hs of the block's tile (bf16: half h of k-group kg, hs = 2 kg + h, see swzk), LDS-DMA'd
// straight into buffer `buf` (no registers): 8 wave-instructions of 1 KB per thread.  Each
// wave-instruction's LDS destination is lane-linear (base + 16 lane), so the A swizzle is applied on
// the per-lane SOURCE address (and undone on the read):
//   A image [BM rows][8 chunks of 16 B], chunk c at slot c ^ swzk((row >> 1) & 7)
//   B image [BN/16 tiles][2 sp][64 lanes][16 B]: the lane's fragment of MFMA sp
// F8 (W8A8): one FULL k-group per stage (16 fp8 = 16 B per chunk): A chunk c = 2 g + s2 holds
// X8[row][128 kg + 32 g + 16 s2 .. + 16), B the fp8 tiled block [s2][lane][16 B] of the tile
// (ops.tile_weight_fp8) -- the same stage images as a bf16 half k-group.
// W8 (W8A16): one FULL k-group per stage -- X as the two bf16 half-k-group A images (each as
// above) and B the fp8 tiled k-group of every tile verbatim ([tile][s2][lane][16 B]: block s2 = h
// holds the lane's k 32 g + 16 h .. + 16, both sub-steps of half h), converted to bf16 fragments on
// the LDS read -- no quantised copy of X, half the weight bytes of bf16.
// rows (grouped launches): X rows of this thread's pieces (< 0: none)
template <class C, bool WT, bool F8, bool W8 = false, bool GRP = false, bool LINES = true>
VWA_DEVICE void issue_stage(const GemmParams& p, __amdgpu_buffer_rsrc_t rx, __amdgpu_buffer_rsrc_t rw, int bm,
                            int bn, int hs, char* buf, const int (&rows)[C::BM / 8 / C::NW]) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int kg = F8 || W8 ? hs : hs >> 1;
#pragma unroll
  for (int hh = 0; hh < (W8 ? 2 : 1); ++hh) {  // (W8: both bf16 half images of the k-group)
  const int ha = W8 ? hh : F8 ? 0 : hs & 1;
#pragma unroll
  for (int it = 0; it < C::BM / 8 / C::NW; ++it) {
    const int q = it * C::NW + w;  // wave-instruction index: rows 8q .. 8q + 7
    const int r = 8 * q + (lane >> 3), c = (lane & 7) ^ (LINES && !F8 && !W8 ? swzk((r >> 1) & 7) : swz((r >> 1) & 7));
    const int m = GRP ? rows[it] : bm + r;
    unsigned off;
    if constexpr (F8)
      off = (unsigned)((size_t)m * p.ldx + (size_t)kg * BKG + 32 * (c >> 1) + 16 * (c & 1));
    else if constexpr (W8 || !LINES)  // (k 32 g + 16 ha + 8 sp)
      off = (unsigned)(((size_t)m * p.ldx + (size_t)kg * BKG + 32 * (c >> 1) + 16 * ha + 8 * (c & 1)) * 2);
    else
      off = (unsigned)(((size_t)m * p.ldx + (size_t)kg * BKG + 64 * ha + 8 * c) * 2);
    dma16(rx, buf + hh * C::A_BYTES + q * 1024, (GRP ? m >= 0 : m < p.M) ? off : kPastEnd);
  }
  }
  const int kgn = p.K / BKG;
  const int h = F8 || W8 ? 0 : hs & 1;
  if constexpr (W8) {  // the fp8 blocks of the whole k-group, [tile][s2][lane][16 B]
#pragma unroll
    for (int it = 0; it < C::BN / 8 / C::NW; ++it) {
      const int q = it * C::NW + w, T = (bn >> 4) + (q >> 1);
      const unsigned off = T * 16 < p.N ? (unsigned)(((size_t)T * kgn + kg) * 2048 + (q & 1) * 1024 + lane * 16) : kPastEnd;
      dma16(rw, buf + 2 * C::A_BYTES + q * 1024, off);
    }
    return;
  }
#pragma unroll
  for (int it = 0; it < C::BN / 8 / C::NW; ++it) {
    const int q = it * C::NW + w;  // tile q >> 1, sub-step s' = q & 1
    const int tile = q >> 1, sp = q & 1;
    unsigned off;
    if constexpr (F8) {
      const int T = (bn >> 4) + tile;
      off = T * 16 < p.N ? (unsigned)(((size_t)T * kgn + kg) * 2048 + sp * 1024 + lane * 16) : kPastEnd;
    } else if constexpr (WT) {
      const int T = (bn >> 4) + tile;
      const int at = LINES ? (2 * sp + (lane >> 5)) * 512 + h * 256 + (lane & 31) * 8 : (2 * h + sp) * 512 + lane * 8;
      off = T * 16 < p.N ? (unsigned)((((size_t)T * kgn + kg) * 2048 + at) * 2) : kPastEnd;
    } else {
      const int n = bn + tile * 16 + (lane & 15), g = lane >> 4;
      const int at = LINES ? 64 * h + 8 * chunk_of(g, sp) : 32 * g + 16 * h + 8 * sp;
      off = n < p.N ? (unsigned)(((size_t)n * p.K + (size_t)kg * BKG + at) * 2) : kPastEnd;
    }
    dma16(rw, buf + C::A_BYTES + q * 1024, off);
  }
}

// 16 bytes of a stage.  All reads of stages are loads of one vector type: HIP's uint4 is a struct, whose copy says nothing of types,
// and in front of such a read of LDS the compiler waits for every LDS-DMA in flight (vmcnt(0)) -- each stage's first read drained
// what the counted wait above it had left in flight.  fp8 weights, 32 rows: 4096 x 4096 in one slice 30.7 -> 17.7 us, 28672 x 4096
// 35.1 -> 23.1; in eight 4096 x 14336 22.4 -> 17.6 (with their sum).  W8A8 on the 128-row tile: 80 x 4096 x 14336 22.0 -> 20.4,
// 2048 x 8192 at 1100 rows 40.2 -> 38.6.
VWA_DEVICE u32x4 stage16(const char* at) {
  const u32x4 v = *reinterpret_cast<const u32x4*>(at);
  return v;
}

template <class C, bool F8, bool W8 = false, bool LINES = true>
VWA_DEVICE void compute_stage(const char* buf, f32x4 (&acc)[C::FM][C::FN], int wm, int wn) {
  const int l = lane_id();
  const int rl = l & 15, g = l >> 4;
  const char* la = buf + (wm * C::FM * 16 + rl) * 128;
  const char* lb = buf + C::A_BYTES + (wn * C::FN) * 2048 + l * 16;
  if constexpr (W8) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
    // 16 e4m3 per lane and tile (both sub-steps of half h), read once; the per-row weight scale is
    // applied to the finished column in the epilogue
    u32x4 w8[C::FN];
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
      w8[j] = stage16(buf + 2 * C::A_BYTES + (wn * C::FN + j) * 2048 + h * 1024 + l * 16);
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) {
      bf16x8 a[C::FM], b[C::FN];
      const int ch = ((2 * g + sp) ^ swz(rl >> 1)) << 4;
#pragma unroll
      for (int i = 0; i < C::FM; ++i) a[i] = *reinterpret_cast<const bf16x8*>(la + h * C::A_BYTES + i * 16 * 128 + ch);
#pragma unroll
      for (int j = 0; j < C::FN; ++j) {
        const unsigned d0 = sp ? w8[j].z : w8[j].x, d1 = sp ? w8[j].w : w8[j].y;
        uint4 bw;
        bw.x = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, 1.0f, false));
        bw.y = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d0, 1.0f, true));
        bw.z = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, 1.0f, false));
        bw.w = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d1, 1.0f, true));
        b[j] = as_bf16x8(bw);
      }
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
    }
    }
  } else if constexpr (F8) {
    // one 128-deep MX MFMA per fragment pair: lane (row / column, g) supplies the 32 fp8 of
    // k 32 g .. 32 g + 32 -- A chunks 2 g and 2 g + 1 of the swizzled image, B blocks s2 = 0, 1 of
    // the fp8 tiled layout -- each read with one ds_read_b128 (conflict-free, as the bf16 path).
    // (The earlier 16x16x32 form read 8-byte halves, which the compiler merged into
    // ds_read2st64_b64 -- 16-lane groups on 32 banks: 49.8 % LDS bank conflicts,
    // profiles/r3_pmc_fp8_chain.md -- and ran at the bf16 MFMA rate.)
    i32x8 a[C::FM], b[C::FN];
    const int c0 = ((2 * g) ^ swz(rl >> 1)) << 4, c1 = ((2 * g + 1) ^ swz(rl >> 1)) << 4;
#pragma unroll
    for (int i = 0; i < C::FM; ++i) {
      const u32x4 lo = stage16(la + i * 16 * 128 + c0);
      const u32x4 hi = stage16(la + i * 16 * 128 + c1);
      a[i] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    }
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
      const u32x4 lo = stage16(lb + j * 2048);
      const u32x4 hi = stage16(lb + j * 2048 + 1024);
      b[j] = i32x8{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    }
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int j = 0; j < C::FN; ++j) acc[i][j] = mfma16x128_fp8(a[i], b[j], acc[i][j]);
  } else {
#pragma unroll
    for (int sp = 0; sp < 2; ++sp) {
      bf16x8 a[C::FM], b[C::FN];
      // ((row >> 1) & 7) == rl >> 1 for every fragment row
      const int ch = (LINES ? chunk_of(g, sp) ^ swzk(rl >> 1) : (2 * g + sp) ^ swz(rl >> 1)) << 4;
#pragma unroll
      for (int i = 0; i < C::FM; ++i) a[i] = *reinterpret_cast<const bf16x8*>(la + i * 16 * 128 + ch);
#pragma unroll
      for (int j = 0; j < C::FN; ++j) b[j] = *reinterpret_cast<const bf16x8*>(lb + j * 2048 + sp * 1024);
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) acc[i][j] = mfma16(a[i], b[j], acc[i][j]);
    }
  }
}

// ---- 256 x 256 tile, 8 waves (2 x 4, each 128 x 64).  A stage (one bf16 half k-group, 64 deep) is four half-tile
// images of 16 KB -- A-lo (rows 0-63 and 128-191: the first half of either M half), A-hi (the other rows), B-lo (n-tiles
// 0-7), B-hi (8-15) -- in the same layouts as the 128^2 kernel, and runs as two phases of 32 MFMAs per wave: A reads all
// of the wave's B fragments and its four fragments of A-lo, B those of A-hi (the B fragments stay in registers).  A phase is operand reads and DMA issue; waits;
// barrier; MFMAs; barrier -- and the two wave groups (M halves) run one barrier apart, so that one group's reads overlap
// the other group's MFMAs.  What bounds it is the time a phase adds to its MFMAs (barriers, the tail of the LDS reads):
// with four phases of 16 MFMAs and the DMA addresses computed per stage the matrix cores were busy 58 % of 4096 x 8192 x
// 8192.
//   DMA: the halves of a buffer are refilled as they fall free, two stages ahead: A-lo, B-lo and B-hi of stage s + 2 in
//   phase B of stage s (all read in phase A), A-hi of stage s + 1 in phase A of stage s (read in phase B of s - 1); the
//   two wave instructions of a half-tile need no vector address math (the stage is the scalar offset).  Each phase waits
//   until 8 instructions are left, which covers what the next phase reads: both groups have passed that wait by the
//   barrier after which the first of them reads it.  A group's reads are retired (lgkmcnt) before the barrier that lets
//   the other one refill what they read.
// Measured (TFLOP/s, four phases with 32-byte X pieces -> two phases -> whole lines): 4096 x 8192 x 8192 1194 -> 1297 ->
// 1425, 2048 x 4096 x 22528 1106 -> 1226 -> 1329, 1011 x 28672 x 4096 SwiGLU 1020 -> 1217 -> 1244.
using CfgP8 = Cfg<256, 256, 2, 4>;

// ---- 128 x 128 | 192 tile, two groups of 4 waves (each 64 x 64 | 96): products whose tiles are one to a CU at most.  Four waves
// alone in a CU read a stage, multiply it and wait for the next by turns (1.27 us per k-group where two workgroups to a CU take 0.92
// each; three and four stages ahead, or eight waves on the same stage, are 0 - 5 % faster).  Here group g takes the stages
// g, g + 2, .. and runs one barrier behind the other: one reads while the other multiplies, and the sums meet in LDS at the end.
//   A group's turn: operand reads; barrier; the next but one stage's DMA into what was read, MFMAs, wait for the next stage; barrier.
//   (A ring of five stages, DMA between the MFMAs: the same.  Both groups at once, with one barrier per two stages: 52 us of
//   the 41 below.  A CU draws 57 bytes a ns then, 64 on the 256^2 tile and 70 at most: the wide tile needs a sixth less of it.)
// us, alone or two to a CU -> two groups: 1011 x 4096 x 4096 48.1 -> 40.9, 2048 x 2048 x 2048 28.2 -> 23.8, 700 x 1280 x 1280 (in
// slices before) 20.6 -> 15.2; 192 columns: 1011 x 6144 x 4096 62.8 -> 54.0, 130 x 12288 x 2048 29.4 -> 24.0.
// Residuals and heads are stored by both groups, in turn, with a row's position and slot requested in front of the LDS round trip and
// its rotation behind the sums: a product into rotated heads and cache, 1011 x 6144 x 4096, 69.5 -> 63.7 us, 600 rows 50.2 -> 47.0.
// (Plain results: no difference.)  What leaves straight from the registers -- 32-bit results, slices -- is half of either group: by one
// group, with 32-bit residuals, 2048 x 1024 x 2048 34.4 -> 28.2, 600 x 2048 x 1536 24.3 -> 20.6, and 1011 x 4096 x 6144 72.2 -> 65.3.
// half-tile `which` (0 A-lo, 1 A-hi, 2 B-lo, 3 B-hi) into the stage image `st`: 16 wave-instructions of 1 KB, 2 per
// wave, from the byte offsets voff (past the resource: zeros) + soff
VWA_DEVICE void p8_issue(__amdgpu_buffer_rsrc_t r, const unsigned (&voff)[8], unsigned soff, int which, char* st) {
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int i = which < 2 ? 2 * it + which : 2 * which + it;
    char* to = st + (which < 2 ? (8 * i + w) * 1024 : CfgP8::A_BYTES + (8 * (i - 4) + w) * 1024);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)to, 16, voff[i], soff, 0, 0);
  }
}

// one phase: 32 MFMAs, acc[i0 .. i0+3][0 .. 3] over both k-substeps of the stage (fp8: 16 of twice the depth)
template <int I0, bool F8>
VWA_DEVICE void p8_mfma(f32x4 (&acc)[8][4], const bf16x8 (&a)[4][2], const bf16x8 (&b)[4][2]) {
  __builtin_amdgcn_s_setprio(1);
  if constexpr (F8) {
    auto both = [](const bf16x8 (&v)[2]) {
      typedef int i32x4 __attribute__((ext_vector_type(4)));
      return __builtin_shufflevector(__builtin_bit_cast(i32x4, v[0]), __builtin_bit_cast(i32x4, v[1]), 0, 1, 2, 3, 4, 5, 6, 7);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[I0 + i][j] = mfma16x128_fp8(both(a[i]), both(b[j]), acc[I0 + i][j]);
  } else
#pragma unroll
  for (int sp = 0; sp < 2; ++sp)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[I0 + i][j] = mfma16(a[i][sp], b[j][sp], acc[I0 + i][j]);
  __builtin_amdgcn_s_setprio(0);
}

VWA_DEVICE float bias_at(const GemmParams& p, int n) { return p.bias ? bf2f(p.bias[n]) : 0.f; }

// RMS statistics hand-off (GemmParams::ss_*): sums of squares in u64 fixed point, 2^-24 units,
// each partial rounded to nearest (truncation biased every atomic add down by up to one unit --
// visible on small-norm rows).  Headroom: 2^64 / 2^24 ~ 1.1e12 per row sum; one partial is
// clamped to 9.2e18 so a handful of them cannot wrap the counter.
constexpr double kSsScale = 16777216.0;
VWA_DEVICE unsigned long long ss_fix(float sq) {
  return (unsigned long long)fminf(sq * (float)kSsScale + 0.5f, 9.2e18f);  // (>= 0)
}

VWA_DEVICE float ss_scale(const GemmParams& p, unsigned long long ss) {
  return rsqrtf((float)((double)ss * (1.0 / kSsScale)) / (float)p.K + p.ss_eps);
}
// per-row RMSNorm scale: rstd[m], or from the handed-off sum of squares (ss_in), or 1
VWA_DEVICE float row_scale(const GemmParams& p, int m) {
  if (p.rstd) return p.rstd[m];
  if (p.ss_in) return ss_scale(p, p.ss_in[m]);
  return 1.f;
}

VWA_DEVICE float resid_at(const GemmParams& p, int m, int n) {
  return p.y_f32 == 2 ? reinterpret_cast<const float*>(p.R)[(size_t)m * p.ldr + n] : bf2f(p.R[(size_t)m * p.ldr + n]);
}

VWA_DEVICE float relu2(float v) {
  v = fmaxf(v, 0.f);
  return v * v;
}

template <int EPI>
VWA_DEVICE void store_out(const GemmParams& p, int m, int n, float v) {
  if constexpr (kResid<EPI>) v += resid_at(p, m, n);
  if (p.y_f32)
    reinterpret_cast<float*>(p.Y)[(size_t)m * p.ldy + n] = v;
  else
    reinterpret_cast<u16*>(p.Y)[(size_t)m * p.ldy + n] = f2bf(v);
}

// EPI_QKV: output chunk n .. n+7 (o) of row m and its rotation partner n^8 (q) -> rotary (q / k
// heads) -> q_out or the paged K / V caches, 16-byte stores.  Within a head (permuted rows) the
// chunk at column 16 t + 8 hi holds dims hi * hd/2 + 8 t .. + 8, its partner the other half.
//   rope: the row's (cos, sin) of the chunk's 8 dims (use_rope); slot: the row's cache slot
VWA_DEVICE const float4* rope_at(const GemmParams& p, int pos, int n) {
  return reinterpret_cast<const float4*>(p.rope + ((size_t)pos * (p.head_dim >> 1) + 8 * ((n % p.head_dim) >> 4)) * 2);
}
VWA_DEVICE void qkv_store(const GemmParams& p, int m, int n, const float (&o)[8], const float (&q)[8],
                          const float4 (&rope)[4], int64_t slot) {
  const int hd = p.head_dim, half = hd >> 1;
  const int head = n / hd, wc = n % hd;
  const int t = wc >> 4;
  const bool hi = (wc & 8) != 0;
  const bool is_v = head >= p.n_q_heads + p.n_kv_heads;
  float y[8];
  if (p.use_rope && !is_v) {
#pragma unroll
    for (int e2 = 0; e2 < 4; ++e2) {
      const float4 v = rope[e2];  // (cos, sin) of dims 2 e2, 2 e2 + 1
      const int e = 2 * e2;
      y[e] = hi ? o[e] * v.x + q[e] * v.y : o[e] * v.x - q[e] * v.y;
      y[e + 1] = hi ? o[e + 1] * v.z + q[e + 1] * v.w : o[e + 1] * v.z - q[e + 1] * v.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = o[e];
  }
  const int d = (hi ? half : 0) + 8 * t;
  if (head < p.n_q_heads) {
    *reinterpret_cast<uint4*>(p.q_out + (size_t)m * p.ldq + head * hd + d) = pack8(y);
    return;
  }
  if (slot < 0) return;
  const int kvh = is_v ? head - p.n_q_heads - p.n_kv_heads : head - p.n_q_heads;
  const int64_t idx = (slot / p.block_size) * p.cache_sb + kvh * p.cache_sh + (slot % p.block_size) * p.cache_st;
  *reinterpret_cast<uint4*>((is_v ? p.v_cache : p.k_cache) + idx + d) = pack8(y);
}

// f32 partial slab loads of the split-K reduce (AUX: buffer cache bits; the reduce runs after the
// GEMM launch's end made the slabs visible, so plain loads)
template <int AUX>
VWA_DEVICE f32x4 ld_f4(__amdgpu_buffer_rsrc_t r, size_t idx) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(idx * 4), 0, AUX));
}

VWA_DEVICE void add8(float (&v)[8], const f32x4& a, const f32x4& b) {
  v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w; v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
}

// Split-K output items: row m, output columns c .. c+7 -- the sum of every slice's f32 partial
// (slice order: the result does not depend on which slice finished last) and the epilogue
// (SwiGLU: features c .. c+7 from the interleaved gate / up columns; QKV: also the rotation
// partner chunk c^8, then rotary + q / KV stores), 16-byte stores.
//   src0 / src1: the item's two 8-column source chunks (SwiGLU gate / up; QKV own / partner)
template <int EPI>
VWA_DEVICE int item_src0(int c) { return EPI == EPI_SWIGLU ? (c >> 4) * 32 + (c & 15) : c; }
template <int EPI>
VWA_DEVICE int item_src1(int c) { return EPI == EPI_SWIGLU ? item_src0<EPI>(c) + 16 : (c ^ 8); }
template <int EPI>
constexpr bool kTwoSrc = EPI == EPI_SWIGLU || EPI == EPI_QKV;

// one item's slices z0 .. z0 + ZB - 1; those past the last read past the slab range (the buffer returns zeros)
template <int EPI, int AUX, int ZB>
struct ItemSlabs {
  f32x4 x[ZB][2], y[kTwoSrc<EPI> ? ZB : 1][2];
  VWA_DEVICE void load(const GemmParams& p, __amdgpu_buffer_rsrc_t rws, int m, int c, int z0) {
    const size_t slab = (size_t)p.M * p.N;
    const int n0 = item_src0<EPI>(c), n1 = item_src1<EPI>(c);
#pragma unroll
    for (int u = 0; u < ZB; ++u) {
      const size_t base = (size_t)(z0 + u) * slab + (size_t)m * p.N;
      x[u][0] = ld_f4<AUX>(rws, base + n0);
      x[u][1] = ld_f4<AUX>(rws, base + n0 + 4);
      if constexpr (kTwoSrc<EPI>) {
        y[u][0] = ld_f4<AUX>(rws, base + n1);
        y[u][1] = ld_f4<AUX>(rws, base + n1 + 4);
      }
    }
  }
  VWA_DEVICE void add(float (&a)[8], float (&b)[8]) const {
#pragma unroll
    for (int u = 0; u < ZB; ++u) {
      add8(a, x[u][0], x[u][1]);
      if constexpr (kTwoSrc<EPI>) add8(b, y[u][0], y[u][1]);
    }
  }
};

// what the epilogue of an item reads besides the slabs, as it was read: nothing here waits for a load (behind the sums each was one more
// dependent round trip, and a reduction of few rows is nothing else)
template <int EPI> struct ItemRaw {
  static constexpr bool kBias = EPI != EPI_SWIGLU;
  int pos;
  int64_t slot;
  float sx;
  unsigned scale[2];  // rstd's value or the two halves of the sum of squares
  f32x4 swa[2], swb[2];
  u32x4 ba, bb;    // 8 bf16
  u32x4 r0, r1;    // residual: 8 bf16 (r0) or f32 (vectors: as structs they went through 272 bytes of scratch a lane)
};
// (parts of a caller's tensors: aligned as their elements)
typedef u32x4 u32x4_bf __attribute__((aligned(2)));
typedef f32x4 f32x4_f __attribute__((aligned(4)));
VWA_DEVICE u32x4 ld_bf8(const u16* q) { return *reinterpret_cast<const u32x4_bf*>(q); }
VWA_DEVICE void ld_f8(const float* q, f32x4 (&v)[2]) {
  v[0] = *reinterpret_cast<const f32x4_f*>(q);
  v[1] = *reinterpret_cast<const f32x4_f*>(q + 4);
}
template <int EPI>
VWA_DEVICE ItemRaw<EPI> item_raw(const GemmParams& p, int m, int c) {
  ItemRaw<EPI> q;
  const int n0 = item_src0<EPI>(c), n1 = item_src1<EPI>(c);
  q.pos = EPI == EPI_QKV && p.use_rope ? p.positions[m] : 0;
  q.slot = EPI == EPI_QKV ? p.slots[m] : 0;
  q.sx = p.sx ? p.sx[m] : 1.f;
  q.scale[0] = q.scale[1] = 0;
  if (p.rstd || p.ss_in) {
    const unsigned* s = p.rstd ? reinterpret_cast<const unsigned*>(p.rstd + m) : reinterpret_cast<const unsigned*>(p.ss_in + m);
    q.scale[0] = s[0];
    q.scale[1] = s[p.rstd ? 0 : 1];
  }
  q.swa[0] = q.swa[1] = q.swb[0] = q.swb[1] = f32x4{1.f, 1.f, 1.f, 1.f};
  q.ba = q.bb = q.r0 = q.r1 = u32x4{0, 0, 0, 0};
  if (p.sw) {
    ld_f8(p.sw + n0, q.swa);
    if constexpr (kTwoSrc<EPI>) ld_f8(p.sw + n1, q.swb);
  }
  if (ItemRaw<EPI>::kBias && p.bias) {
    q.ba = ld_bf8(p.bias + n0);
    if constexpr (EPI == EPI_QKV) q.bb = ld_bf8(p.bias + n1);
  }
  const bool wide = p.y_f32 == 2;                    // f32 residual stream: 16-byte accesses (rows are 32-byte aligned)
  if (wide || (kResid<EPI> && !p.y_f32)) {
    const char* r = reinterpret_cast<const char*>(p.R) + ((size_t)m * p.ldr + c) * (wide ? 4 : 2);
    q.r0 = *reinterpret_cast<const u32x4*>(r);
    q.r1 = *reinterpret_cast<const u32x4*>(r + (wide ? 16 : 0));
  }
  return q;
}
// ... made ready, under the slabs' loads or behind them
template <int EPI> struct ItemPre {
  float scale, swa[8], swb[8], ba[8], bb[8];
  u32x4 r0, r1;
  f32x4 rope[4];
  int64_t slot;
};
template <int EPI>
VWA_DEVICE ItemPre<EPI> item_ready(const GemmParams& p, const ItemRaw<EPI>& r, const f32x4 (&rope)[4]) {
  ItemPre<EPI> q;
  unsigned lo = r.scale[0], hi = r.scale[1];
  asm volatile("" : "+v"(lo), "+v"(hi));             // (else the conversion, and a wait, follow the loads into their branch)
  q.scale = (p.rstd ? __uint_as_float(lo) : p.ss_in ? ss_scale(p, (unsigned long long)hi << 32 | lo) : 1.f) * r.sx;
#pragma unroll
  for (int e = 0; e < 8; ++e) q.swa[e] = r.swa[e >> 2][e & 3], q.swb[e] = r.swb[e >> 2][e & 3];
  unpack8(__builtin_bit_cast(uint4, r.ba), q.ba);
  unpack8(__builtin_bit_cast(uint4, r.bb), q.bb);
  q.r0 = r.r0;
  q.r1 = r.r1;
  q.slot = r.slot;
#pragma unroll
  for (int e = 0; e < 4; ++e) q.rope[e] = rope[e];
  return q;
}

// epilogue of one summed item + its stores
// returns the sum of squares of the stored bf16 values (residual epilogue with ss_out; else 0)
template <int EPI>
VWA_DEVICE float finish_item(const GemmParams& p, const ItemPre<EPI>& q, int m, int c, const float (&a)[8], float (&b)[8]) {
  const float rs = q.scale;
  float v[8];
  if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = silu(a[e] * q.swa[e] * rs) * (b[e] * q.swb[e] * rs);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = a[e] * rs * q.swa[e] + q.ba[e];
      if constexpr (kGelu<EPI>) v[e] = gelu_erf(v[e]);
    }
    if constexpr (EPI == EPI_QKV) {
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = b[e] * rs * q.swb[e] + q.bb[e];
      float4 rope[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) rope[e] = __builtin_bit_cast(float4, q.rope[e]);
      qkv_store(p, m, c, v, b, rope, q.slot);
      return 0.f;
    }
  }
  if constexpr (EPI == EPI_SPLIT) {
    if (c >= p.n_split) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = relu2(v[e]);
      *reinterpret_cast<uint4*>(p.Y2 + (size_t)m * p.ldy2 + c - p.n_split) = pack8(v);
      return 0.f;
    }
  }
  if (p.y_f32 == 2) {
    float4* y = reinterpret_cast<float4*>(reinterpret_cast<float*>(p.Y) + (size_t)m * p.ldy + c);
    const float4 r0 = __builtin_bit_cast(float4, q.r0), r1 = __builtin_bit_cast(float4, q.r1);
    y[0] = make_float4(v[0] + r0.x, v[1] + r0.y, v[2] + r0.z, v[3] + r0.w);
    y[1] = make_float4(v[4] + r1.x, v[5] + r1.y, v[6] + r1.z, v[7] + r1.w);
    return 0.f;
  }
  if (p.y_f32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) store_out<EPI>(p, m, c + e, v[e]);
    return 0.f;
  }
  if constexpr (kResid<EPI>) {
    float r[8];
    unpack8(__builtin_bit_cast(uint4, q.r0), r);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += r[e];
  }
  const uint4 o = pack8(v);
  *reinterpret_cast<uint4*>(reinterpret_cast<u16*>(p.Y) + (size_t)m * p.ldy + c) = o;
  float sq = 0.f;
  if (kResid<EPI> && p.ss_out) {
    unpack8(o, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) sq += v[e] * v[e];
  }
  return sq;
}

// ss_out[m] += sq summed over the wave's lanes of each row (lanes with m < 0 add nothing): one
// atomic per row per wave when the wave lies in one row, else one per lane
VWA_DEVICE void ss_add(unsigned long long* ss_out, int m, float sq) {
  const int m0 = __builtin_amdgcn_readfirstlane(m);
  if (__ballot(m != m0) == 0ull) {
    sq = wave_sum(sq);
    if (lane_id() == 0 && m0 >= 0)
      __hip_atomic_fetch_add(gp(ss_out + m0), ss_fix(sq), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else if (m >= 0) {
    __hip_atomic_fetch_add(gp(ss_out + m), ss_fix(sq), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Few rows: everything the item reads is in flight together, the rotary row behind its position.  (With the scale, the bias and the
// rotary row each waited for ahead of the slabs, us of the launch: 8 rows of 1280 columns with bias and residual 5.0 -> 4.0, 32 rows of
// 4096, 8 slices, 5.0 -> 4.7, of 6144 with the rotation 5.0 -> 4.8.)
template <int EPI, int AUX, int ZB>
VWA_DEVICE float reduce_item(const GemmParams& p, __amdgpu_buffer_rsrc_t rws, int m, int c) {
  float a[8] = {}, b[8] = {};
  const ItemRaw<EPI> q = item_raw<EPI>(p, m, c);
  ItemSlabs<EPI, AUX, ZB> s;
  s.load(p, rws, m, c, 0);
  asm volatile("" ::: "memory");
  f32x4 rope[4] = {};
  if (EPI == EPI_QKV && p.use_rope) {
    const f32x4* at = reinterpret_cast<const f32x4*>(rope_at(p, q.pos, c));
#pragma unroll
    for (int e = 0; e < 4; ++e) rope[e] = at[e];
    asm volatile("" ::: "memory");
  }
  const ItemPre<EPI> pre = item_ready<EPI>(p, q, rope);
  s.add(a, b);
  for (int z0 = ZB; z0 < p.splits; z0 += ZB) {
    s.load(p, rws, m, c, z0);
    s.add(a, b);
  }
  return finish_item<EPI>(p, pre, m, c, a, b);
}

// (a 4-stage variant for one-row-block GEMMs measured slower in whole decode steps -- 128 KB
// of LDS leaves one workgroup per CU, so split-K grids above 256 workgroups ran in two rounds:
// fp8 32 rows 4.97 vs 4.36 ms, profiles/r4_gemm_ab.md -- and was removed)
template <class C, int EPI, bool WT, bool F8 = false, bool P8 = false, bool W8 = false, bool GRP = false, bool LINES = !GRP>
__global__ __launch_bounds__(C::THREADS, C::NW == 4 ? 2 : 1) void gemm_kernel(GemmParams p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int FM = C::FM, FN = C::FN;
  static_assert(!GRP || (WT && !F8 && !W8 && (EPI == EPI_SWIGLU || EPI == EPI_STORE)), "grouped: tiled bf16");
  const int mb = GRP ? p.g_tiles[0] : (p.M + C::BM - 1) / C::BM, nb = (p.N + C::BN - 1) / C::BN;
  const int tiles = mb * nb;
  // (few rows' launches are over in 8 us, and the compiler's divisions are a chain of 25 operations each in front of the first load)
  const bool small = gridDim.x < (unsigned)kSmallDiv;
  const int part = gridDim.x == (unsigned)tiles ? 0 : small ? small_div(blockIdx.x, tiles) : blockIdx.x / tiles;
  const int split = p.nbatch > 1 ? 0 : part;  // split-K slice (blocks of one slice are contiguous)
  if (p.nbatch > 1) {  // batch z = blockIdx.x / tiles, splits == 1 (vwa_gemm)
    const int z = part;
    p.X += (size_t)z * p.bsx;
    p.Y = reinterpret_cast<char*>(p.Y) + (size_t)z * p.bsy * (p.y_f32 ? 4 : 2);
    if (p.R) p.R += (size_t)z * p.bsr;
  }
  // XCD-aware: logical tile order is column-block major, so consecutive logical tiles (same XCD)
  // share the column block's weight tile in L2
  if (p.ss_zero && blockIdx.x == 0)
    for (int i = threadIdx.x; i < p.ss_zero_n; i += C::THREADS) p.ss_zero[i] = 0ull;
  if (GRP && (int)blockIdx.x >= tiles) return;       // (the grid is sized for the most row blocks there can be)
  const int lt = xcd_remap((int)blockIdx.x - part * tiles, tiles);
  // (grouped: column blocks of kGroup row blocks -- mostly one expert's -- after one another)
  const int band = GRP ? lt / (kGroup * nb) * kGroup : 0, bh = GRP ? min(kGroup, mb - band) : mb, bt = lt - band * nb;
  const int col = bh == 1 ? bt : small ? small_div(bt, bh) : bt / bh, row = bt - col * bh;
  const int bn = col * C::BN;
  int bm = row * C::BM, place = 0;
  int rows[C::BM / 8 / C::NW];
  size_t x_rows = 0;
  if constexpr (GRP) {
    const int gt = band + row;
    p.W += (size_t)p.g_tiles[1 + 3 * gt] * p.g_wstride;
    place = p.g_tiles[2 + 3 * gt];
    x_rows = (size_t)p.M;                            // (X rows the buffer holds)
    p.M = p.g_tiles[3 + 3 * gt];
    bm = 0;
#pragma unroll
    for (int it = 0; it < C::BM / 8 / C::NW; ++it) {
      const int r = 8 * (it * C::NW + (threadIdx.x >> 6)) + ((threadIdx.x & 63) >> 3);
      rows[it] = r < p.M ? (p.g_down ? place + r : p.g_order[place + r] / p.g_top) : -1;
    }
  }
  const int KG = p.K / BKG;
  const int kg0 = split * p.kg_per_split, kg1 = min(KG, kg0 + p.kg_per_split);
  const int w = C::GROUPS > 1 ? (threadIdx.x >> 6) % C::NW : threadIdx.x >> 6, wm = w / C::WN, wn = w % C::WN;
  const int grp = C::GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * C::NW)) : 0;
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // pipeline: NST LDS buffers, the next NST - 1 stages' DMA in flight during this one's MFMAs; raw
  // barriers with counted vmcnt (a __syncthreads would drain the in-flight DMA)
  constexpr int SPG = F8 || W8 ? 1 : 2;  // stages per k-group
  constexpr int STG = W8 ? C::W8STAGE : C::STAGE;
  constexpr int NST = W8 ? C::W8NST : C::NST;  // stage buffers
  constexpr int PER = (W8 ? 2 : 1) * (C::BM / 8 / C::NW) + C::BN / 8 / C::NW;  // LDS-DMA instructions of a stage and wave
  static_assert(PER * (NST - 1) < 64, "LDS-DMA instructions of the stages in flight (the counted vmcnt)");
  const int h0 = SPG * kg0, nh = SPG * (kg1 - kg0);
  // X extent: the last row starts at (M-1)*ldx and is K long (rows may overlap: conv views)
  const size_t x_bytes = ((GRP ? x_rows - 1 : (size_t)(p.M - 1)) * p.ldx + p.K) * (F8 ? 1 : 2);
  const size_t w_bytes = (size_t)p.N * p.K * (F8 || W8 ? 1 : 2);
  const __amdgpu_buffer_rsrc_t rx = rsrc(p.X, x_bytes), rw = rsrc(p.W, w_bytes);
  if constexpr (P8) {
    static_assert(C::BM == 256 && C::BN == 256 && C::NW == 8, "two-phase pipeline: CfgP8");
    constexpr bool PAIRS = F8 || !LINES;  // a lane group's two chunks side by side (k 32 g ..), not by whole cache lines
    const int l = lane_id(), rl = l & 15, g = l >> 4;
    auto stage = [&](int s) { return lds + (s & 1) * C::STAGE; };
    unsigned voff[8];  // this lane's pieces of the half-tiles (k-group 0)
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int q = it * 8 + w, r = 8 * q + (l >> 3), m = GRP ? rows[it] : bm + r;  // A rows 8 q ..
      voff[it] = (GRP ? m >= 0 : m < p.M) ? p8_x_piece<F8, LINES>(m, p.ldx, r, l) : kPastEnd;
      const int T = (bn >> 4) + (q >> 1);  // B n-tile q / 2, MFMA q & 1
      voff[4 + it] = T * 16 < p.N ? p8_w_piece<F8, WT, LINES>(T, q & 1, p.K, l) : kPastEnd;
    }
    // (stages past the last are issued too, on empty resources: the waits stay one constant)
    auto issue = [&](int s, int which) {
      const bool in = s < nh;
      if (which < 2)
        p8_issue(rsrc(p.X, in ? x_bytes : 0), voff, p8_x_step<F8, LINES>(h0 + s, in), which, stage(s));
      else
        p8_issue(rsrc(p.W, in ? w_bytes : 0), voff, p8_w_step<F8, WT, LINES>(h0 + s, in), which, stage(s));
    };
    issue(0, 0);
    issue(0, 2);
    issue(0, 3);
    issue(0, 1);
    issue(1, 0);
    issue(1, 2);
    issue(1, 3);
    asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    bf16x8 a[4][2], b[4][2];
    if (wm == 1) asm volatile("s_barrier" ::: "memory");  // group 1 runs one barrier behind group 0
    for (int s = 0; s < nh; ++s) {
      const char* st = stage(s);
      const char* la = st + (wm * 128 + rl) * 128;
      const char* lb = st + C::A_BYTES + (wn * 4) * 2048 + l * 16;
      auto read_a = [&](int i0) {
#pragma unroll
        for (int sp = 0; sp < 2; ++sp)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            a[i][sp] = *reinterpret_cast<const bf16x8*>(la + (i0 + i) * 16 * 128 + ((PAIRS ? (2 * g + sp) ^ swz(rl >> 1) : chunk_of(g, sp) ^ swzk(rl >> 1)) << 4));
      };
#pragma unroll
      for (int sp = 0; sp < 2; ++sp)
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j][sp] = *reinterpret_cast<const bf16x8*>(lb + j * 2048 + sp * 1024);
      read_a(0);
      issue(s + 1, 1);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      p8_mfma<0, F8>(acc, a, b);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_barrier" ::: "memory");
      read_a(4);
      issue(s + 2, 0);
      issue(s + 2, 2);
      issue(s + 2, 3);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      p8_mfma<4, F8>(acc, a, b);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_barrier" ::: "memory");
    }
    if (wm == 0) asm volatile("s_barrier" ::: "memory");  // (group 1 started one barrier later)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // (the epilogue reuses the LDS)
  } else if constexpr (C::GROUPS == 2) {
    static_assert(C::NST == 2 && !F8 && !W8 && !GRP && LINES, "two K groups: bf16 products that keep no order");
    const int l = lane_id(), rl = l & 15, g = l >> 4, n = nh / 2;
    constexpr int PA = C::BM / 8 / C::NW, PB = C::BN / 8 / C::NW;
    char* const mine = lds + grp * 2 * C::STAGE;
    unsigned xoff[PA], woff[PB];  // this lane's pieces of a stage (k-group 0)
#pragma unroll
    for (int it = 0; it < PA; ++it) {
      const int r = 8 * (it * C::NW + w) + (l >> 3), m = bm + r;
      xoff[it] = m < p.M ? p8_x_piece<F8, LINES>(m, p.ldx, r, l) : kPastEnd;
    }
#pragma unroll
    for (int it = 0; it < PB; ++it) {
      const int q = it * C::NW + w, T = (bn >> 4) + (q >> 1);
      woff[it] = T * 16 < p.N ? p8_w_piece<F8, WT, LINES>(T, q & 1, p.K, l) : kPastEnd;
    }
    // this group's stage i (past the last: on empty resources, so that the waits stay one constant)
    auto issue = [&](int i) {
      const bool in = i < n;
      const int s = h0 + 2 * i + grp;
      char* to = mine + (i & 1) * C::STAGE + w * 1024;
      const __amdgpu_buffer_rsrc_t ra = rsrc(p.X, in ? x_bytes : 0), rb = rsrc(p.W, in ? w_bytes : 0);
      const unsigned sa = p8_x_step<F8, LINES>(s, in), sb = p8_w_step<F8, WT, LINES>(s, in);
#pragma unroll
      for (int it = 0; it < PA; ++it) dma16(ra, to + it * C::NW * 1024, xoff[it], sa);
#pragma unroll
      for (int it = 0; it < PB; ++it) dma16(rb, to + C::A_BYTES + it * C::NW * 1024, woff[it], sb);
    };
    issue(0);
    issue(1);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PER) : "memory");
    if (grp == 1) asm volatile("s_barrier" ::: "memory");
    for (int i = 0; i < n; ++i) {
      const char* st = mine + (i & 1) * C::STAGE;
      const char* la = st + (wm * FM * 16 + rl) * 128;
      const char* lb = st + C::A_BYTES + (wn * FN) * 2048 + l * 16;
      bf16x8 a[FM][2], b[FN][2];
#pragma unroll
      for (int sp = 0; sp < 2; ++sp) {
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j][sp] = *reinterpret_cast<const bf16x8*>(lb + j * 2048 + sp * 1024);
#pragma unroll
        for (int j = 0; j < FM; ++j) a[j][sp] = *reinterpret_cast<const bf16x8*>(la + j * 16 * 128 + ((chunk_of(g, sp) ^ swzk(rl >> 1)) << 4));
      }
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (read by all of the group: free)
      issue(i + 2);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int sp = 0; sp < 2; ++sp)
#pragma unroll
        for (int ii = 0; ii < FM; ++ii)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[ii][j] = mfma16(a[ii][sp], b[j][sp], acc[ii][j]);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PER) : "memory");  // (the next stage has landed)
    }
    if (grp == 0) asm volatile("s_barrier" ::: "memory");  // (group 1 started one barrier later)
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    f32x4* ex = reinterpret_cast<f32x4*>(lds) + w * FM * FN * 64 + l;
    if (p.splits > 1 || p.y_f32) {  // stored from the registers: half of the rows by either group
#pragma unroll
      for (int i = 0; i < FM; ++i)
        if (i / (FM / 2) != grp)
#pragma unroll
          for (int j = 0; j < FN; ++j) ex[(i * FN + j) * 64] = acc[i][j];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < FM; ++i)
        if (i / (FM / 2) == grp)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] += ex[(i * FN + j) * 64];
    } else {
      if (grp == 1) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) ex[(i * FN + j) * 64] = acc[i][j];
      }
      __syncthreads();
      if (grp == 0) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] += ex[(i * FN + j) * 64];
      }
      __syncthreads();  // (the epilogue writes LDS again)
      if (grp == 1 && !(kResid<EPI> || EPI == EPI_QKV)) return;  // (these store by both groups)
    }
  } else {
  if (nh > 0) issue_stage<C, WT, F8, W8, GRP, LINES>(p, rx, rw, bm, bn, h0, lds, rows);
  if (nh > 1) issue_stage<C, WT, F8, W8, GRP, LINES>(p, rx, rw, bm, bn, h0 + 1, lds + STG, rows);
  if (NST > 2 && nh > 2) issue_stage<C, WT, F8, W8, GRP, LINES>(p, rx, rw, bm, bn, h0 + 2, lds + 2 * STG, rows);
  if (NST > 3 && nh > 3) issue_stage<C, WT, F8, W8, GRP, LINES>(p, rx, rw, bm, bn, h0 + 3, lds + 3 * STG, rows);
  static_assert(NST <= 4, "stages issued ahead");
  for (int i = 0; i < nh; ++i) {
    char* at = lds + (NST == 2 || NST == 4 ? i & (NST - 1) : i % NST) * STG;
    // this stage landed everywhere (the ones behind it stay in flight)
    if (NST > 3 && i + 3 < nh)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * PER) : "memory");
    else if (NST > 2 && i + 2 < nh)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * PER) : "memory");
    else if (i + 1 < nh)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PER) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    compute_stage<C, F8, W8, LINES>(at, acc, wm, wn);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave done reading it
    if (i + NST < nh) issue_stage<C, WT, F8, W8, GRP, LINES>(p, rx, rw, bm, bn, h0 + i + NST, at, rows);
  }
  }
  const int l = lane_id();
  const int col0 = bn + wn * FN * 16 + (l & 15);
  const int row0 = bm + wm * FM * 16 + 4 * (l >> 4);
  if (p.splits > 1) {  // f32 partial slab of this slice; gemm_reduce_kernel applies the epilogue
    float* ws = p.ws + (size_t)split * p.M * p.N;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = row0 + i * 16 + r;
        if (m >= p.M || (C::GROUPS > 1 && i / (FM / 2) != grp)) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int n = col0 + j * 16;
          if (n < p.N) ws[(size_t)m * p.N + n] = acc[i][j][r];
        }
      }
    return;
  }
  // per-lane epilogue operands loaded once (no load-or-constant select per element)
  float bz[FN], cz[FN], rsv[FM][4];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    bz[j] = 0.f;
    cz[j] = 1.f;
  }
  if (p.bias) {
#pragma unroll
    for (int j = 0; j < FN; ++j) bz[j] = col0 + j * 16 < p.N ? bf2f(p.bias[col0 + j * 16]) : 0.f;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) rsv[i][r] = 1.f;
  if (p.rstd || p.ss_in) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        rsv[i][r] = row0 + i * 16 + r < p.M ? row_scale(p, GRP ? p.g_order[place + row0 + i * 16 + r] : row0 + i * 16 + r) : 1.f;
  }
  // W8A8: acc * sx[m] * sw[n] (SwiGLU: gate / up columns scale before the activation); W8A16: sw only
  if constexpr (F8 || W8) {
    if constexpr (F8) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) rsv[i][r] *= row0 + i * 16 + r < p.M ? p.sx[row0 + i * 16 + r] : 1.f;
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) cz[j] = col0 + j * 16 < p.N ? p.sw[col0 + j * 16] : 0.f;
  }
  if (p.y_f32) {  // f32 logits (rare: prefill LM head rows) -- direct stores
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = row0 + i * 16 + r;
        if (m >= p.M || (C::GROUPS > 1 && i / (FM / 2) != grp)) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int n = col0 + j * 16;
          if (n >= p.N) continue;
          float v = acc[i][j][r] * rsv[i][r] * cz[j] + bz[j];
          if constexpr (kGelu<EPI>) v = gelu_erf(v);
          if constexpr (kResid<EPI>) v += resid_at(p, m, n);
          reinterpret_cast<float*>(p.Y)[(size_t)m * p.ldy + n] = v;
        }
      }
    return;
  }
  // bf16 results that something is done to behind the product -- the residual added, heads rotated: through LDS in 32 bits,
  // PI fragment rows at a time, and rounded once, as the slices' sum does (rounded in front of it too, a residual of the
  // product's size: 2.15e-3 from float64 instead of 1.66e-3).  A pass's residual chunks are requested in front of its LDS round
  // trip: 1500 x 1280 x 1280 19.7 -> 17.6 us, 12000 x 1280 x 1280 41.2 -> 39.0.  W8A8 products keep both roundings: their
  // results choose fp8 codes further on, and stay as they were.
  if constexpr (!F8 && (kResid<EPI> || EPI == EPI_QKV)) {
    constexpr int CPR = FN * 2, RSF = FN * 64 + 16;  // 8-column chunks of a row; LDS row stride (bytes: 4 rows apart, 16 banks)
    constexpr int LDSB = (W8 ? C::W8LDS : C::LDS) / C::NW / (16 * RSF);
    constexpr int PI = LDSB >= FM ? FM : LDSB >= FM / 2 ? FM / 2 : FM / 4, ITS = PI * 16 * CPR / 64 / C::GROUPS;
    static_assert(PI >= 1 && PI <= LDSB && FM % PI == 0 && (C::GROUPS == 1 || PI == FM), "a pass fits the wave's share of the LDS");
    char* wl = lds + w * (PI * 16 * RSF);
#pragma unroll
    for (int i0 = 0; i0 < FM; i0 += PI) {
      const int mw = bm + (wm * FM + i0) * 16, nw = bn + wn * FN * 16;
      auto row_of = [&](int it) { return ((it * C::GROUPS + grp) * 64 + l) / CPR; };  // (two groups: in turn)
      auto chunk_at = [&](int it) { return ((it * C::GROUPS + grp) * 64 + l) % CPR; };
      uint4 rv[ITS];
      if constexpr (kResid<EPI>) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
          const int m = mw + row_of(it), n = nw + chunk_at(it) * 8;
          if (m < p.M && n < p.N) rv[it] = *reinterpret_cast<const uint4*>(p.R + (size_t)m * p.ldr + n);
        }
      }
      int posv[ITS];
      int64_t slotv[ITS];
      if constexpr (EPI == EPI_QKV) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
          const int m = min(mw + row_of(it), p.M - 1);
          posv[it] = p.use_rope ? p.positions[m] : 0;
          slotv[it] = p.slots[m];
        }
      }
      if (grp == 0)
#pragma unroll
      for (int i = 0; i < PI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            float v = acc[i0 + i][j][r] * rsv[i0 + i][r] * cz[j] + bz[j];
            if constexpr (kGelu<EPI>) v = gelu_erf(v);
            *reinterpret_cast<float*>(wl + (i * 16 + 4 * (l >> 4) + r) * RSF + (j * 16 + (l & 15)) * 4) = v;
          }
      constexpr bool AHEAD = EPI == EPI_QKV && ITS <= 6;  // (the sums' registers are free now)
      float4 turn[AHEAD ? ITS : 1][4];
      if constexpr (AHEAD) {
        if (p.use_rope) {
#pragma unroll
          for (int it = 0; it < ITS; ++it)
#pragma unroll
            for (int e = 0; e < 4; ++e) turn[it][e] = rope_at(p, posv[it], min(nw + chunk_at(it) * 8, p.N - 8))[e];
        }
      }
      if constexpr (C::GROUPS > 1) __syncthreads();
      else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      float sqv[ITS];  // (ss_out: squares of each stored chunk)
#pragma unroll
      for (int it = 0; it < ITS; ++it) {
        sqv[it] = 0.f;
        const int m = mw + row_of(it), n = nw + chunk_at(it) * 8;
        if (m >= p.M || n >= p.N) continue;
        const char* row = wl + row_of(it) * RSF;
        auto chunk = [&](int ch, float (&f)[8]) {
          const float4 a = *reinterpret_cast<const float4*>(row + ch * 32), b = *reinterpret_cast<const float4*>(row + ch * 32 + 16);
          f[0] = a.x, f[1] = a.y, f[2] = a.z, f[3] = a.w, f[4] = b.x, f[5] = b.y, f[6] = b.z, f[7] = b.w;
        };
        float v[8], u[8];
        chunk(chunk_at(it), v);
        if constexpr (EPI == EPI_QKV) {
          chunk(chunk_at(it) ^ 1, u);
          if constexpr (AHEAD) {
            qkv_store(p, m, n, v, u, turn[it], slotv[it]);
          } else {
            float4 rope[4];
            if (p.use_rope) {
#pragma unroll
              for (int e = 0; e < 4; ++e) rope[e] = rope_at(p, posv[it], n)[e];
            }
            qkv_store(p, m, n, v, u, rope, slotv[it]);
          }
        } else {
          unpack8(rv[it], u);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += u[e];
          const uint4 o = pack8(v);
          if (p.ss_out) {
            unpack8(o, u);  // (the stored bf16 values)
#pragma unroll
            for (int e = 0; e < 8; ++e) sqv[it] += u[e] * u[e];
          }
          *reinterpret_cast<uint4*>(reinterpret_cast<u16*>(p.Y) + (size_t)m * p.ldy + n) = o;
        }
      }
      static_assert(!kResid<EPI> || 64 % CPR == 0, "a row's lanes side by side");
      if (kResid<EPI> && p.ss_out) {  // one atomic per (row, wave): the CPR lanes of a row reduce first
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
          const int m = mw + row_of(it);
          float sq = sqv[it];
#pragma unroll
          for (int o = 1; o < CPR; o <<= 1) sq += __shfl_xor(sq, o, 64);
          if (l % CPR == 0 && m < p.M && bn + wn * FN * 16 < p.N)
            __hip_atomic_fetch_add(gp(p.ss_out + m), ss_fix(sq), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    return;
  }
  // bf16 out: the wave's tile goes through LDS (padded rows: the four row groups of a store hit
  // different banks) and leaves as 16-byte row chunks -- coalesced stores, 16-byte residual reads
  constexpr int NCOL = EPI == EPI_SWIGLU ? FN * 8 : FN * 16;  // output columns of this wave
  constexpr int RS = NCOL * 2 + (NCOL == 32 ? 32 : 16);       // LDS row stride (bytes, 16-aligned)
  constexpr int ROWS = FM * 16;
  char* wl = lds + w * (ROWS * RS);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int rl = i * 16 + 4 * (l >> 4) + r;
      if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
        for (int j = 0; j < FN; j += 2) {
          const float gt = acc[i][j][r] * rsv[i][r] * cz[j], up = acc[i][j + 1][r] * rsv[i][r] * cz[j + 1];
          *reinterpret_cast<u16*>(wl + rl * RS + ((j >> 1) * 16 + (l & 15)) * 2) = f2bf(silu(gt) * up);
        }
      } else {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          float v = acc[i][j][r] * rsv[i][r] * cz[j] + bz[j];
          if constexpr (kGelu<EPI>) v = gelu_erf(v);
          if constexpr (EPI == EPI_SPLIT) v = col0 + j * 16 >= p.n_split ? relu2(v) : v;  // (uniform per fragment)
          *reinterpret_cast<u16*>(wl + rl * RS + (j * 16 + (l & 15)) * 2) = f2bf(v);
        }
      }
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int CPR = NCOL / 8;  // 16-byte chunks per row
  const int ncols = EPI == EPI_SWIGLU ? p.N / 2 : p.N;
  const int cbase = EPI == EPI_SWIGLU ? (bn + wn * FN * 16) / 2 : bn + wn * FN * 16;
  float sqv[ROWS * CPR / 64];  // (ss_out: squares of each stored chunk)
#pragma unroll
  for (int it = 0; it < ROWS * CPR / 64; ++it) {
    sqv[it] = 0.f;
    const int idx = it * 64 + l, row = idx / CPR, ch = idx % CPR;
    const int m = bm + wm * ROWS + row, n = cbase + ch * 8;
    if (m >= p.M || n >= ncols) continue;
    uint4 v = *reinterpret_cast<const uint4*>(wl + row * RS + ch * 16);
    if constexpr (EPI == EPI_QKV) {  // (bf16-rounded like the stored projection it replaces)
      float o[8], q[8];
      unpack8(v, o);
      unpack8(*reinterpret_cast<const uint4*>(wl + row * RS + (ch ^ 1) * 16), q);
      float4 rope[4];
      if (p.use_rope) {
        const int pos = p.positions[m];
#pragma unroll
        for (int e = 0; e < 4; ++e) rope[e] = rope_at(p, pos, n)[e];
      }
      qkv_store(p, m, n, o, q, rope, p.slots[m]);
      continue;
    }
    if constexpr (kResid<EPI>) {
      float a[8], b[8];
      unpack8(v, a);
      unpack8(*reinterpret_cast<const uint4*>(p.R + (size_t)m * p.ldr + n), b);
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] += b[e];
      v = pack8(a);
      if (p.ss_out) {
        unpack8(v, a);  // (the stored bf16 values)
#pragma unroll
        for (int e = 0; e < 8; ++e) sqv[it] += a[e] * a[e];
      }
    }
    if (EPI == EPI_SPLIT && n >= p.n_split)
      *reinterpret_cast<uint4*>(p.Y2 + (size_t)m * p.ldy2 + n - p.n_split) = v;
    else
      *reinterpret_cast<uint4*>(reinterpret_cast<u16*>(p.Y) + (size_t)(GRP ? (p.g_down ? p.g_order[place + m] : place + m) : m) * p.ldy + n) = v;
  }
  if (kResid<EPI> && p.ss_out) {  // one atomic per (row, wave): the CPR lanes of a row reduce first
#pragma unroll
    for (int it = 0; it < ROWS * CPR / 64; ++it) {
      const int idx = it * 64 + l, row = idx / CPR, ch = idx % CPR;
      const int m = bm + wm * ROWS + row;
      float sq = sqv[it];
#pragma unroll
      for (int o = 1; o < CPR; o <<= 1) sq += __shfl_xor(sq, o, 64);  // the CPR lanes of one row
      if (ch == 0 && m < p.M && cbase < ncols)
        __hip_atomic_fetch_add(gp(p.ss_out + m), ss_fix(sq), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// sum of the split-K slabs + epilogue (two-launch split-K): one thread per (row, 8 output columns), ZB slices in flight
template <int EPI, int ZB>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmParams p) {
  const int cpr = (EPI == EPI_SWIGLU ? p.N / 2 : p.N) / 8;
  const int64_t id = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool ok = id < (int64_t)p.M * cpr;
  const __amdgpu_buffer_rsrc_t rws = rsrc(p.ws, (size_t)p.splits * p.M * p.N * 4);
  float sq = 0.f;
  const int m = (int)((unsigned)id / (unsigned)cpr);  // (M N fits 32-bit slab offsets)
  if (ok) sq = reduce_item<EPI, 0, ZB>(p, rws, m, (int)((unsigned)id - (unsigned)m * cpr) * 8);
  if (kResid<EPI> && p.ss_out) ss_add(p.ss_out, ok ? m : -1, sq);
}

// per-row 1/rms of X (the RMSNorm of a projection whose gamma is folded into W)
__global__ __launch_bounds__(256) void row_rstd_kernel(const u16* __restrict__ x, int ldx, int M, int K, float eps,
                                                       float* __restrict__ rstd) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const u16* xr = x + (size_t)row * ldx;
  float ss = 0.f;
  for (int c = lane_id() * 8; c < K; c += 64 * 8) {
    float f[8];
    unpack8(*reinterpret_cast<const uint4*>(xr + c), f);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += f[j] * f[j];
  }
  ss = wave_sum(ss);
  if (lane_id() == 0) rstd[row] = rsqrtf(ss / (float)K + eps);
}

int cdiv(int a, int b) { return (a + b - 1) / b; }

// bf16 weights on tile C
template <class C, int EPI>
int launch_cfg(const GemmParams& p, hipStream_t st) {
  const int tiles = ((p.M + C::BM - 1) / C::BM) * ((p.N + C::BN - 1) / C::BN);
  const dim3 grid(tiles * p.splits * (p.nbatch > 1 ? p.nbatch : 1));
  if (p.w_tiled)
    hipLaunchKernelGGL((gemm_kernel<C, EPI, true, false>), grid, dim3(C::THREADS), C::LDS, st, p);
  else
    hipLaunchKernelGGL((gemm_kernel<C, EPI, false, false>), grid, dim3(C::THREADS), C::LDS, st, p);
  return 0;
}

// a product that keeps its order of sums, on any tile
template <class C, int EPI, bool P8>
void launch_kept(const GemmParams& p, hipStream_t st) {
  hipLaunchKernelGGL((gemm_kernel<C, EPI, true, false, P8, false, false, false>), dim3(cdiv(p.M, C::BM) * cdiv(p.N, C::BN) * p.splits),
                     dim3(C::THREADS), C::LDS, st, p);
}

int g_p8_mode = 2;         // 0: the 128^2 kernel only, 1: the 256^2 one from 256 rows (bf16: of pre-tiled whole column tiles), 2: choose()
int g_split_fill_pct = 0;  // > 0: vwa_gemm_splits' fill, and the rules by shape alone instead of plan()

// Whether a product may take the two-group tile of n columns: pre-tiled bf16 weights whose sums keep no order (the two groups' are
// added last).  65 .. 127 rows, whose slices are by shape alone, keep the other tile and their bits: of 10 weights at 85 rows one
// gained (28672 x 4096 62.9 -> 58.7 us) and one lost (6144 x 4096 24.3 -> 24.8).  The wide one has 12 chunks to a row, which the residual's epilogue does not deal out.
constexpr bool takes_wide(int epi) { return epi != EPI_RESID && epi != EPI_GELU_RESID; }
bool takes_groups(const GemmParams& p, int epi, int n) {
  return g_p8_mode == 2 && p.w_tiled && !p.sw && !p.keep_order && p.nbatch <= 1 && p.cus > 0 && p.M >= 128 && (n == CfgK::BN || takes_wide(epi));
}

// Tile and K slices of a bf16 product of >= 128 rows: the cheapest by an estimate in us, fitted to 180 shapes (130 .. 12000
// rows, 384 .. 28672 columns, K 384 .. 14336; both tiles, 1 .. 16 slices): 9 % off (rms of the logarithm), and 1.4 % slower than the
// best choice of each shape, where the rules before (256^2 from 256 tiles or from slices of >= 2048 k that fill the CUs;
// slices in powers of two until 75 % of the CUs have a tile) were 12 %: 12000 x 1280 x 5120 (235 large tiles) 165 -> 115 us,
// 768 x 4096 x 14336 155 -> 86, 512 x 28672 x 4096 132 -> 93, 1863 x 6144 x 4096 115 -> 83.
//   a round of the CUs costs so much per k-group and so much to start and store; a part of a last round 70 % and its share;
//   128^2 tiles run two to a CU, one alone is faster, two groups on one (CfgK, CfgKw) faster still wherever every tile has a CU;
//   beyond that tiles by twos are (1024 x 8192 x 2048, 512 tiles: 41 us, 48 of two groups);
//   the slices' f32 partials are written and read.
//   Two groups have fewer k-groups each to pay for their start and the meeting of their sums: from 8 of a slice on (over 131 products of
//   5 .. 7 they were 1.4 % slower, 1.14 times at worst), from 11 where one row block has the weight to itself (128 rows: 8 and 10 up to
//   1.08 times).  192 columns in slices must be 5 % ahead by the estimate: taken at any lead, 29 of 70 such products were slower.  Of 728
//   products with other tiles than without groups: 8.0 % less time on average, 12 are 2 - 4.5 % slower (profiles/gemm_tiles_ab.csv).
//   A residual in 32 bits is added element by element behind whole tiles, 8 us on two groups and 14 on one, which the sum of slices does
//   not pay: its product has the slices that it would have on one-group tiles (2048 x 1024 x 2048 whole 28.2 us, two slices 25.6 on one
//   group).
// W8A8 (k-groups of half the stages): fitted to 690 timings of 60 shapes (80 .. 6000 rows, 1024 .. 28672 columns, K 1280 ..
// 14336), 11 % off; it picks the tile alone: slices in another order move a few bf16 activations by a bit, and every moved one
// can flip its fp8 code further on, so they stay those of vwa_gemm_splits.  2720 x 4096 x 14336 224 -> 125 us, 2720 x 28672 x
// 4096 407 -> 294, 1863 x 6144 x 4096 75 -> 48; small ones keep the 128^2 tile (2720 x 2560 x 1280: 18.4, 24.7 on the large one).
// tile: columns of the small tile taken (CfgK: with a minus)
float estimate(const GemmParams& p, bool p8, int s, int epi, int* tile = nullptr) {
  const int kg = cdiv(p.K / BKG, s), b = p8 ? 256 : 128;
  const int64_t t = (int64_t)cdiv(p.M, b) * cdiv(p.N, b) * s;
  const bool alone = !p8 && t <= p.cus;
  const float r = (float)t / (p8 || alone ? p.cus : 2 * p.cus), whole = floorf(r);
  const float rounds = r <= 1.f ? 1.f : r > whole ? whole + 0.7f + 0.3f * (r - whole) : whole;
  const float slabs = (float)s * p.M * p.N * 4.f;
  if (p.sx) {
    const float per = p8 ? 1.21f : alone ? 0.97f : r >= 1.f ? 1.17f : 0.97f + 0.2f * (2.f * r - 1.f);
    return rounds * (kg * per + (p8 ? 6.8f : 3.3f)) + (s > 1 ? 5.3f + slabs / 3.27e6f : 0.f);
  }
  const float per = p8 ? 2.0f : alone ? 1.27f : r >= 1.f ? 1.84f : 1.27f + 0.57f * (2.f * r - 1.f);
  const float sum = s > 1 ? 4.f + slabs / 3.55e6f : 0.f;
  float us = rounds * (kg * per + (p8 ? 5.6f : 2.3f));
  if (!p8) {
    if (tile) *tile = CfgS::BN;
    float least = us;
    for (const int n : {CfgK::BN, CfgKw::BN}) {
      if (!takes_groups(p, epi, n) || kg < (p.M <= CfgK::BM ? 11 : 8) || (int64_t)cdiv(p.M, CfgK::BM) * cdiv(p.N, n) * s > p.cus) continue;
      const float g = n == CfgK::BN ? kg * 0.99f + 3.6f : s == 1 ? kg * 1.18f + 5.f : 1.05f * (kg * 1.18f + 5.f) + 0.05f * sum;
      if (g < least) {
        least = g;
        if (tile) *tile = n == CfgK::BN ? -CfgK::BN : CfgKw::BN;
      }
    }
    if (p.y_f32 != 2 || s > 1) us = least;
  }
  return us + sum;
}

struct Plan {
  bool p8;
  int splits;
};
Plan plan(const GemmParams& p, int epi, float* took = nullptr) {
  const int KG = p.K / BKG;
  Plan best{false, 1};
  float least = 0.f;
  for (const int s0 : {1, 2, 3, 4, 6, 8, 12, 16}) {
    if (s0 > 1 && (s0 > KG || (int64_t)s0 * p.M * p.N > p.ws_cap)) break;
    for (const bool p8 : {true, false}) {
      const float us = estimate(p, p8, cdiv(KG, cdiv(KG, s0)), epi);
      if (least == 0.f || us < least) {
        least = us;
        best = {p8, s0};
      }
    }
  }
  if (took) *took = least;
  return best;
}

// Whether the kernels' 32-bit offsets reach all of a product's weight and rows (loads past a resource's end are zeros)
bool reachable(const GemmParams& p) {
  constexpr int64_t kMost = 0x7FFFFFF0ll;
  return (int64_t)p.N * p.K * (p.sw ? 1 : 2) < kMost && ((int64_t)(p.M - 1) * p.ldx + p.K) * (p.sx ? 1 : 2) < kMost;
}

// Columns of a product that fill whole rounds of the CUs with large tiles, where it is cheaper by the estimate to give the rest a
// launch of its own, with tiles and slices of its own (0: not).  The tiles past the last whole round cost nearly a round of their
// own, however few: 2048 x 32896 x 4096 is four rounds and eight tiles, 482 -> 438 us in two launches (398 of them the whole rounds').
// 1024 x 17664 x 2048 86 -> 76 us, 1300 x 22528 x 4096 238 -> 206, 1900 x 26624 x 4096 341 -> 333.  182 products that are cut: 10 % less
// time on average, one (850 x 17664 x 2048, whose one-group tiles fill two rounds) 4 - 7 % more (profiles/gemm_tiles_ab.csv).
int whole_rounds(const GemmParams& p, int epi) {
  if (!reachable(p)) return 0;  // (one launch, which refuses it whole)
  if (p.M < 128 || p.keep_order || p.sw || p.nbatch > 1 || p.cus <= 0 || g_p8_mode != 2 || g_split_fill_pct != 0) return 0;
  const int mb = cdiv(p.M, 256), nb = cdiv(p.N, 256), tiles = mb * nb;
  const int cols = mb <= p.cus ? (int)((int64_t)(tiles / p.cus) * p.cus / mb) : 0;  // column tiles of the whole rounds
  if (cols < 1 || cols * 256 >= p.N) return 0;
  float whole, rest;
  plan(p, epi, &whole);
  GemmParams a = p, b = p;
  a.N = cols * 256;
  b.N = p.N - a.N;
  plan(b, epi, &rest);
  return estimate(a, true, 1, epi) + rest + 3.f < 0.97f * whole ? a.N : 0;
}

// K slices of a bf16 product of <= 64 rows and of fp8 weights (W8A16): the cheapest by an estimate in us, fitted to 270 timings
// (24, 48 and 64 rows, 22 weights of 1024 .. 32768 columns and K 1024 .. 14336, 1 .. 32 slices) and for fp8 weights to 520.
//   a workgroup's k-groups one after another, against all of the weight at the chip's rate (the larger counts, both where they are
//   close); a sum of slices is a launch and its f32 partials
// bf16: priced at one number of rows, so that the weight alone decides and a row's sums are added up in one order whatever rows
// come with it.  Over 28 weights in the tiles taken now, 1, 16, 32, 48, 64 rows, slower than the best choice of each by
//   priced at 48 rows           2.3, 3.8, 6.5, 3.8, 5.5 %      at the rows of the call  6.4, 4.8, 7.2, 3.8, 5.8 %
//   the same for the norm, at 1 0.9, 1.1, 1.5, 0.2, 0.1 %                               1.0, 2.8, 4.6, 4.0, 5.0 %
// fp8 weights at the rows of the call (0.8, 0.5, 0.5, 1.2 % at 17, 32, 48, 64 rows; priced at 24 rows they would be 0.7, 1.0, 1.0,
// 0.6 %, but rows summed in another order flip fp8 codes in the products of <= 16 rows behind them: logits of a 48-row prompt on
// 1024-wide layers move by 0.03, with the same 0.028 from 64 bits).
// Powers of two until the CUs have a tile are 6 % (bf16) and 10 % (fp8) off and up to 50 % where one slice fills half the chip (48
// rows: 17664 x 2048 26.3 us in two slices, 20.3 whole; fp8, 32 rows: 28672 x 4096 30.0 in two, 23.1 whole).
// parts: no launch adds the slices up, but the workgroup of a row's norm reads its row of each (at about 40 GB/s)
int few_slices(const GemmParams& p, bool parts) {
  const int KG = p.K / BKG, blocks = cdiv(p.M, CfgF::BM);
  const bool w8 = p.sw != nullptr;
  const int M = w8 ? p.M : parts ? 1 : 48, most = w8 ? p.M : CfgF::BM;
  const float per_kg = w8 ? (M <= CfgFs::BM ? 0.42f : 0.68f) + 0.00065f * (blocks > 1 ? CfgF::BM : M) : 0.52f + 0.0063f * M;
  const float chip = (float)p.N * p.K * blocks * (w8 ? 1.f / 6.2e6f : 2.f / 6.1e6f) * (256.f / p.cus);
  const float launch = w8 ? 2.6f : 3.2f, slab = (float)M * p.N * (4 * (w8 ? 0.53e-6f : 0.44e-6f));
  int best = 1;
  float least = 0.f;
  for (int s0 = 1; s0 <= 32 && s0 <= KG; s0 *= 2) {
    if (s0 > 1 && (int64_t)s0 * most * p.N > p.ws_cap) break;
    const int per = cdiv(KG, s0), s = cdiv(KG, per);
    const float alone = per_kg * per;
    const float sum = parts ? (float)s * p.N * (4 / 4.e4f) : s > 1 ? launch + s * slab : 0.f;
    const float us = cbrtf(alone * alone * alone + chip * chip * chip) + sum;
    if (s0 == 1 || us < least) {
      least = us;
      best = s0;
    }
  }
  return best;
}

// Slices of whole large tiles by shape alone, in powers of two until they cover the CUs; *fill: the tiles alone, or slices of
// >= 2048 k each, do
int slices_256(const GemmParams& p, bool* fill) {
  const int tiles = cdiv(p.M, 256) * (p.N / 256);
  int s = 1;
  while (tiles * s < p.cus && s * 2 <= p.K / BKG && (int64_t)(s * 2) * p.M * p.N <= p.ws_cap) s *= 2;
  *fill = tiles >= 256 || (tiles * s >= p.cus && p.K / s >= 2048);
  return s;
}

bool keeps_order(int epi, const GemmParams& p) {
  return p.keep_order && p.w_tiled && !p.sw && p.nbatch <= 1 && p.cus > 0 && (epi == EPI_STORE || epi == EPI_SWIGLU);
}

// Tile and slices of a launch (p.splits: those of vwa_gemm_splits; p.ws_cap: the f32 numbers that slices may take)
Plan choose(const GemmParams& p, int epi, bool parts = false) {
  Plan r{false, p.splits < 1 ? 1 : p.splits};
  if (p.nbatch > 1 || p.cus <= 0) return r;
  if (p.sw && !p.sx) {
    if (g_split_fill_pct == 0) r.splits = few_slices(p, false);
    return r;
  }
  bool fill = false;
  const int s = p.M >= 256 && p.N % 256 == 0 ? slices_256(p, &fill) : 0;
  // (g_p8_mode picks the tile; the slices of W8A8 and kept-order products are part of the order of their sums)
  if (p.keep_order || p.sx) {
    if (p.keep_order && fill) r.splits = s;
    r.p8 = g_p8_mode == 1 ? p.M >= 256 : g_p8_mode == 2 && (p.sx || p.M >= 128) && estimate(p, true, r.splits, epi) < estimate(p, false, r.splits, epi);
    return r;
  }
  if (g_p8_mode == 2 && g_split_fill_pct == 0) {
    if (p.M <= CfgF::BM) r.splits = few_slices(p, parts);
    return p.M >= 128 ? plan(p, epi) : r;
  }
  if (p.w_tiled && s && (g_p8_mode == 1 || (g_p8_mode == 2 && fill))) r = Plan{true, s};
  return r;
}

// Tiles of 64 columns: a product of <= 64 rows whose 128-column tiles and slices leave half of the CUs without one: twice as many
// draw weights, each k-group is over sooner, and a row's sums are the same.  us on 128 / 64 columns, 1, 32 and 48 rows: 9472 x 1024
// 9.1 / 7.4, 9.5 / 7.5, 11.2 / 9.3, 16384 x 2048 18.7 / 16.0, 19.0 / 15.4, 20.4 / 16.6, 3072 x 512 5.7 / 4.7, 5.8 / 4.8, 7.0 / 5.9;
// 1.12 - 1.36 times faster on all 17 weights of 1536 .. 16384 columns and K 384 .. 2048, row-major ones 1.18 - 1.59.  In slices, with
// their sum, 16 and 48 rows: 1024 x 4096 8.8 / 8.4, 10.5 / 9.5, 1280 x 1280 7.3 / 6.7, 8.6 / 7.5; 1.03 - 1.17 times on 7 weights.
constexpr bool takes_narrow(int epi) { return epi != EPI_SWIGLU && epi != EPI_GELU_RESID; }
bool narrow(const GemmParams& p) {  // (bf16 weights that keep no order)
  return g_p8_mode == 2 && p.M <= CfgN::BM && p.nbatch <= 1 && 2 * cdiv(p.N, 128) * p.splits <= p.cus;
}

// Columns of the tile of 128 rows that a product of more than 64 takes (CfgK: with a minus)
int small_tile(const GemmParams& p, int epi) {
  int tile = CfgS::BN;
  if (takes_groups(p, epi, CfgK::BN)) estimate(p, false, p.splits, epi, &tile);
  return tile;
}

template <class C, int EPI>
void launch_groups(const GemmParams& p, hipStream_t st) {
  hipLaunchKernelGGL((gemm_kernel<C, EPI, true>), dim3(cdiv(p.M, C::BM) * cdiv(p.N, C::BN) * p.splits), dim3(C::THREADS), C::LDS, st, p);
}

// sum false: the slices' partial rows stay in the workspace
template <int EPI>
int launch_epi(const GemmParams& p, hipStream_t st, bool p8, bool sum = true) {
  constexpr bool kKeeps = EPI == EPI_STORE || EPI == EPI_SWIGLU;
  if (kKeeps && p.keep_order) {
    if constexpr (kKeeps) {
      if (p8) launch_kept<CfgP8, EPI, true>(p, st);
      else if (p.M <= CfgFs::BM) launch_kept<CfgFs, EPI, false>(p, st);
      else if (p.M <= CfgF::BM) launch_kept<CfgF, EPI, false>(p, st);
      else launch_kept<CfgS, EPI, false>(p, st);
    }
  } else if (p8) {
    const int tiles = ((p.M + 255) / 256) * ((p.N + 255) / 256);
    if (p.sx)
      hipLaunchKernelGGL((gemm_kernel<CfgP8, EPI, true, true, true>), dim3(tiles * p.splits), dim3(CfgP8::THREADS),
                         CfgP8::LDS, st, p);
    else if (p.w_tiled)
      hipLaunchKernelGGL((gemm_kernel<CfgP8, EPI, true, false, true>), dim3(tiles * p.splits), dim3(CfgP8::THREADS),
                         CfgP8::LDS, st, p);
    else
      hipLaunchKernelGGL((gemm_kernel<CfgP8, EPI, false, false, true>), dim3(tiles * p.splits), dim3(CfgP8::THREADS),
                         CfgP8::LDS, st, p);
  } else if (p.sw && !p.sx) {  // W8A16 (tiles of 128 columns alone: of 64 they have not been built or timed)
    const dim3 grid((unsigned)(cdiv(p.M, CfgF::BM) * cdiv(p.N, CfgF::BN) * p.splits)), block(CfgF::THREADS);
    if (p.M <= CfgFs::BM)
      hipLaunchKernelGGL((gemm_kernel<CfgFs, EPI, true, false, false, true>), grid, block, CfgFs::W8LDS, st, p);
    else
      hipLaunchKernelGGL((gemm_kernel<CfgF, EPI, true, false, false, true>), grid, block, CfgF::W8LDS, st, p);
  } else if (p.sw) {  // W8A8
    hipLaunchKernelGGL((gemm_kernel<CfgS, EPI, true, true>), dim3(cdiv(p.M, CfgS::BM) * cdiv(p.N, CfgS::BN) * p.splits),
                       dim3(CfgS::THREADS), CfgS::LDS, st, p);
  } else if (takes_narrow(EPI) && narrow(p)) {
    if constexpr (takes_narrow(EPI)) {
      if (p.M <= CfgNs::BM) launch_cfg<CfgNs, EPI>(p, st);
      else launch_cfg<CfgN, EPI>(p, st);
    }
  } else if (p.M <= CfgFs::BM) {  // (a row's sums are those of the 128-row tile, and so are the bits)
    launch_cfg<CfgFs, EPI>(p, st);
  } else if (p.M <= CfgF::BM) {
    launch_cfg<CfgF, EPI>(p, st);
  } else {
    const int tile = small_tile(p, EPI);
    if (tile == -CfgK::BN) {
      launch_groups<CfgK, EPI>(p, st);
    } else if (tile == CfgKw::BN) {
      if constexpr (takes_wide(EPI)) launch_groups<CfgKw, EPI>(p, st);
    } else {
      launch_cfg<CfgS, EPI>(p, st);
    }
  }
  if (sum && p.splits > 1) {
    const int64_t n = (int64_t)p.M * (EPI == EPI_SWIGLU ? p.N / 2 : p.N) / 8;
    // one wave per workgroup up to four per CU: a CU alone draws ~25 GB/s of slabs
    const int t = n <= (int64_t)p.cus * 256 ? 64 : 256;
    const dim3 grid((unsigned)((n + t - 1) / t));
    if (p.splits > 4 && t == 64) hipLaunchKernelGGL((gemm_reduce_kernel<EPI, 8>), grid, dim3(t), 0, st, p);
    else hipLaunchKernelGGL((gemm_reduce_kernel<EPI, 4>), grid, dim3(t), 0, st, p);
  }
  return (int)hipGetLastError();
}

template <class C, int EPI, bool P8>
int launch_grouped(const GemmParams& p, hipStream_t st) {
  const dim3 grid(p.g_max * ((p.N + C::BN - 1) / C::BN)), block(C::THREADS);
  hipLaunchKernelGGL((gemm_kernel<C, EPI, true, false, P8, false, true>), grid, block, C::LDS, st, p);
  return (int)hipGetLastError();
}

}  // namespace

// Split-K slices for a shape: enough workgroups to cover the CUs ~2x when the output tiles
// alone cannot (few rows: weight streaming), bounded by the k-groups and the workspace.
// Split while the workgroups cover less than this % of the CUs (0: per-dtype default).  Measured
// on the Llama-3-8B decode steps of 32 / 64 rows (tools/rows_sweep.py, profiles/r4_gemm_ab.md):
// bf16 75 % (5.08 / 5.69 ms vs 5.21 / 6.08 at 100 %), fp8 100 % (4.42 / 5.03 vs 4.62 / 5.06 at 75 %).
// (bf16 products of >= 128 rows: plan(); of <= 64 rows and W8A16: few_slices())
extern "C" int vwa_gemm_splits(int M, int N, int K, int cus, int64_t ws_floats, int f8) {
  const int tiles = ((M + CfgS::BM - 1) / CfgS::BM) * ((N + CfgS::BN - 1) / CfgS::BN);
  const int KG = K / BKG;
  int s = 1;
  const int pct = g_split_fill_pct > 0 ? g_split_fill_pct : f8 ? 100 : 75;
  const int fill = (int)((int64_t)cus * pct / 100);
  while (tiles * s < fill && s * 2 <= KG && (int64_t)(s * 2) * M * N <= ws_floats) s *= 2;
  return s;
}

extern "C" void vwa_gemm_set_split_fill(int pct) { g_split_fill_pct = pct < 0 ? 0 : pct; }

extern "C" void vwa_gemm_set_p8(int mode) { g_p8_mode = mode; }

extern "C" void vwa_gemm_plan(int epi, const GemmParams* pp, int parts, int* columns, int* splits, int* groups) {
  GemmParams p = *pp;
  p.keep_order = keeps_order(epi, p);
  const Plan pl = choose(p, epi, parts);
  const int per = cdiv(p.K / BKG, pl.splits);
  p.splits = *splits = cdiv(p.K / BKG, per);
  *columns = pl.p8 ? CfgP8::BN : !p.keep_order && !p.sw && takes_narrow(epi) && narrow(p) ? CfgN::BN : CfgS::BN;
  *groups = 1;
  if (!pl.p8 && small_tile(p, epi) != CfgS::BN) {
    *columns = small_tile(p, epi) == CfgKw::BN ? CfgKw::BN : CfgK::BN;
    *groups = CfgK::GROUPS;
  }
}

namespace {
int checks_and_plan(int epi, GemmParams& p, bool* p8, bool parts = false) {
  if (p.M < 1 || p.N < 16 || p.N % 16 || p.K < BKG || p.K % BKG) return -10;
  if (p.ldx % (p.sx ? 16 : 8) || (reinterpret_cast<uintptr_t>(p.X) & 15) || (reinterpret_cast<uintptr_t>(p.W) & 15))
    return -11;
  if (!reachable(p)) return -21;
  if ((p.sw && !p.w_tiled) || (p.sx && !p.sw)) return -14;  // fp8: the tiled layout; X codes need fp8 weights
  if (epi == EPI_SWIGLU && (p.N % 32 || p.y_f32)) return -12;
  if (epi == EPI_QKV && (p.y_f32 || p.head_dim % 16 || p.N != (p.n_q_heads + 2 * p.n_kv_heads) * p.head_dim ||
                         !p.q_out || !p.k_cache || !p.v_cache || !p.slots || (p.use_rope && (!p.rope || !p.positions))))
    return -16;
  if (p.y_f32 == 2 && epi != EPI_RESID) return -18;
  if (epi == EPI_SPLIT && (p.y_f32 || !p.Y2 || p.n_split % 16 || p.n_split < 0 || p.n_split > p.N || p.ldy2 % 8 ||
                           (reinterpret_cast<uintptr_t>(p.Y2) & 15)))
    return -19;
  p.keep_order = keeps_order(epi, p);
  const Plan pl = choose(p, epi, parts);
  *p8 = pl.p8;
  p.splits = pl.splits;
  const int KG = p.K / BKG;
  p.kg_per_split = (KG + p.splits - 1) / p.splits;
  p.splits = (KG + p.kg_per_split - 1) / p.kg_per_split;  // no empty slice
  if (p.splits > 1 && !p.ws) return -13;
  if (p.nbatch > 1 && p.splits > 1) return -15;  // batched launches take no split-K
  return 0;
}
}  // namespace

// Products whose consumer adds the slices up itself, in their order: f32 partial rows [parts][M][N] in p.ws, as many as
// vwa_gemm_plan says (1: the product).  Few rows take many slices (48 x 1024 x 6144: 24 when this was timed), whose sum is a launch of its own and nothing but
// round trips; the norm that reads its result reads the slices instead: sum 5.1 + norm 3.6 -> 5.8 us, whole steps of 48 rows 2.7 %
// less.
extern "C" int vwa_gemm_parts(const GemmParams* pp, int parts, hipStream_t st) {
  GemmParams p = *pp;
  bool p8 = false;
  p.Y = p.ws;
  p.ldy = p.N;
  p.y_f32 = 1;
  if (!p.ws || p.bias || p.rstd || p.ss_in || p.sx || p.nbatch > 1) return -10;
  const int r = checks_and_plan(EPI_STORE, p, &p8, true);
  if (r) return r;
  if (p.splits != parts) return -20;  // (ws holds another number of rows)
  return launch_epi<EPI_STORE>(p, st, p8, false);
}

extern "C" int vwa_gemm(int epi, const GemmParams* pp, hipStream_t st) {
  GemmParams p = *pp;
  bool p8 = false;
  if (const int r = checks_and_plan(epi, p, &p8)) return r;
  switch (epi) {
    case EPI_STORE: return launch_epi<EPI_STORE>(p, st, p8);
    case EPI_RESID: return launch_epi<EPI_RESID>(p, st, p8);
    case EPI_SWIGLU: return launch_epi<EPI_SWIGLU>(p, st, p8);
    case EPI_GELU: return launch_epi<EPI_GELU>(p, st, p8);
    case EPI_GELU_RESID: return launch_epi<EPI_GELU_RESID>(p, st, p8);
    case EPI_QKV: return launch_epi<EPI_QKV>(p, st, p8);
    case EPI_SPLIT: return launch_epi<EPI_SPLIT>(p, st, p8);
    default: return -3;
  }
}

// The first n columns of a product whose columns two launches share (vwa_gemm_cut), and the others
extern "C" void vwa_gemm_part(int epi, const GemmParams* pp, int n, int second, GemmParams* part) {
  GemmParams p = *pp;
  if (!second) {
    p.N = n;
    p.n_split = p.n_split < n ? p.n_split : n;
  } else {
    const int out = epi == EPI_SWIGLU ? n / 2 : n;
    p.N -= n;
    p.W += (size_t)n * p.K;
    if (p.bias) p.bias += n;
    if (p.R) p.R += p.y_f32 == 2 ? 2 * out : out;
    if (epi == EPI_SPLIT) {
      if (n > p.n_split) p.Y2 += n - p.n_split;
      p.n_split = p.n_split > n ? p.n_split - n : 0;
    }
    p.Y = reinterpret_cast<char*>(p.Y) + (size_t)out * (p.y_f32 ? 4 : 2);
    p.ss_zero = nullptr;
  }
  *part = p;
}

extern "C" int vwa_gemm_cut(int epi, const GemmParams* pp) {
  GemmParams p = *pp;
  p.keep_order = keeps_order(epi, p);
  return epi == EPI_STORE || epi == EPI_RESID || epi == EPI_SWIGLU || epi == EPI_GELU || epi == EPI_SPLIT ? whole_rounds(p, epi) : 0;
}

extern "C" int vwa_gemm_grouped(int epi, const GemmParams* pp, hipStream_t st) {
  GemmParams p = *pp;
  if (p.M < 1 || p.N % 16 || p.N < 16 || p.K < BKG || p.K % BKG || p.ldx % 8 || p.ldy % 8 || p.y_f32 || p.bias || p.R || p.sw || p.sx ||
      p.ss_in || p.ss_out || p.ss_zero || !p.w_tiled || p.nbatch > 1 || !p.g_tiles || !p.g_order || p.g_max < 1 || p.g_top < 1)
    return -10;
  if ((reinterpret_cast<uintptr_t>(p.X) | reinterpret_cast<uintptr_t>(p.W) | reinterpret_cast<uintptr_t>(p.Y)) & 15) return -11;
  if (epi == EPI_SWIGLU && (p.N % 32 || !p.rstd)) return -12;
  if ((int64_t)p.M * p.ldx * 2 >= 0x7FFFFFF0ll || (int64_t)p.N * p.K * 2 >= 0x7FFFFFF0ll) return -13;  // (32-bit offsets)
  p.splits = 1;
  p.nbatch = 1;
  p.kg_per_split = p.K / BKG;
  if (epi != EPI_SWIGLU && epi != EPI_STORE) return -3;
  if (p.g_tile == CfgS::BM) return epi == EPI_SWIGLU ? launch_grouped<CfgS, EPI_SWIGLU, false>(p, st) : launch_grouped<CfgS, EPI_STORE, false>(p, st);
  if (p.g_tile == CfgP8::BM) return epi == EPI_SWIGLU ? launch_grouped<CfgP8, EPI_SWIGLU, true>(p, st) : launch_grouped<CfgP8, EPI_STORE, true>(p, st);
  return -4;
}

extern "C" int vwa_row_rstd(const uint16_t* x, int ldx, int M, int K, float eps, float* rstd, hipStream_t st) {
  if (M < 1 || K % 8 || ldx % 8) return -1;
  hipLaunchKernelGGL(row_rstd_kernel, dim3((M + 3) / 4), dim3(256), 0, st, x, ldx, M, K, eps, rstd);
  return (int)hipGetLastError();
}
