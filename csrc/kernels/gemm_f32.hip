// 32-bit GEMM on the f32 MFMA (v_mfma_f32_16x16x4_f32: f32 products, f32 accumulation) for models
// that run in 32-bit: Y = epi(X . W^T), both operands row-major with K contiguous.
//
// A lane's 16-byte operand holds 4 consecutive k of its row; the four MFMAs of a 16-deep step take
// element j of every lane group, so A and B use the same k order.  Two kernels (launch() chooses):
//   * rows: a workgroup owns 16 or 32 columns and up to 64 rows, its waves split K and add up through
//     LDS.  Few rows stream the weights, so what counts is bytes in flight on every CU: the k split
//     gives a 1024-column projection 64 x 16 waves of them.
//   * tiles: 64 x 64 outputs, operands by LDS-DMA, for products bound by the MFMA.
// A row's sums have one order for a weight, whatever rows come with it (a token's result, and the expert it
// is sent to, does not depend on how it is batched): K in 32-deep slices, the slices in 8 or 16 runs
// (runs_log2: by N and K alone), a run's products one after the other, a quarter's runs in order, then
// the quarters.
#include "common.h"
#include "stack_kernels.h"

using namespace vwa;

namespace {

VWA_DEVICE f32x4 mfma4(float a, float b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

VWA_DEVICE f32x4 mfma4x4(const float4& a, const float4& b, f32x4 c) {
  c = mfma4(a.x, b.x, c);
  c = mfma4(a.y, b.y, c);
  c = mfma4(a.z, b.z, c);
  return mfma4(a.w, b.w, c);
}

// rows m .. m+3 of column n (EPI 2: v0 gate and v1 up of feature n)
template <int EPI>
VWA_DEVICE void store4(const GemmF32Params& p, int m, int n, const f32x4& v0, const f32x4& v1) {
  if (n >= (EPI == 2 ? p.N >> 1 : p.N)) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (m + r >= p.M) return;
    float v = v0[r];
    if constexpr (EPI == 2) v = silu(v) * v1[r];
    if constexpr (EPI == 1) v += p.R[(size_t)(m + r) * p.ldr + n];
    if (EPI == 6 && n >= p.n_split) {
      v = fmaxf(v, 0.f);
      p.Y2[(size_t)(m + r) * p.ldy2 + n - p.n_split] = v * v;
    } else {
      p.Y[(size_t)(m + r) * p.ldy + n] = v;
    }
  }
}

// Bound by the weights' stream: 4 x 1024 x 4096 12.6 us (1.3 TB/s from 64 workgroups; 122 with one wave per 32 x 32
// outputs), 4 x 8192 x 1024 9.6 us (3.5 TB/s; 38), 4 x 32768 x 1024 30 us (4.5 TB/s; 50).
// 16 MT rows x 16 NT columns; the NW waves take one or two of K's KS runs each, U 16-deep steps' loads in
// flight while the U before are multiplied.
// QR: one quarter of the runs to a workgroup (blockIdx.z), its sum to rows of its own p.part further on: the norm behind the
// product adds the quarters in the order in which they are added up here.  Four times the workgroups for products of few columns: 4 x 1024 x
// 4096 13.5 -> 6.6 us, 4 x 1024 x 1024 5.5 -> 4.8.
template <int EPI, int MT, int NT, int KS, int U, int NW, bool QR = false>
__global__ __launch_bounds__(64 * NW) void rows_f32_kernel(GemmF32Params p) {
  static_assert(!QR || (EPI == 0 && KS == 4 * NW), "a quarter's runs, a wave each");
  __shared__ f32x4 part[(QR ? NW : KS) * MT * NT * 64];
  const int lane = threadIdx.x & 63, w = NW == 16 || MT > 1 ? threadIdx.x >> 6 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rl = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.y * 16 * MT, n0 = blockIdx.x * 16 * NT;
  // rows past the end read the last row (their results are not stored)
  const float* xa[MT];
  const float* wb[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xa[i] = p.X + (size_t)min(m0 + 16 * i + rl, p.M - 1) * p.ldx + 4 * g;
#pragma unroll
  for (int j = 0; j < NT; ++j) wb[j] = p.W + (size_t)min(n0 + 16 * j + rl, p.N - 1) * p.K + 4 * g;
  const int steps = p.K / 16, slices = (steps + 1) / 2;
  f32x4 acc[MT][NT];
  float4 a0[U][MT], b0[U][NT], a1[U][MT], b1[U][NT];
  auto load = [&](float4 (&a)[U][MT], float4 (&b)[U][NT], int s) {
    // (a row's steps after one another: two are a cache line)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int u = 0; u < U; ++u) b[u][j] = *reinterpret_cast<const float4*>(wb[j] + (size_t)(s + u) * 16);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int u = 0; u < U; ++u) a[u][i] = *reinterpret_cast<const float4*>(xa[i] + (size_t)(s + u) * 16);
  };
  auto multiply = [&](const float4 (&a)[U][MT], const float4 (&b)[U][NT]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma4x4(a[u][i], b[u][j], acc[i][j]);
  };
#pragma unroll
  for (int h = 0; h < (QR ? 1 : KS / NW); ++h) {
    const int slot = QR ? w : w * (KS / NW) + h, run = QR ? blockIdx.z * NW + w : slot, s0 = slices * run / KS * 2, n = min(slices * (run + 1) / KS * 2, steps) - s0, full = n / U;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (full > 0) load(a0, b0, s0);
    for (int t = 0; t < full; t += 2) {
      if (t + 1 < full) load(a1, b1, s0 + (t + 1) * U);
      multiply(a0, b0);
      if (t + 1 >= full) break;
      if (t + 2 < full) load(a0, b0, s0 + (t + 2) * U);
      multiply(a1, b1);
    }
    for (int s = s0 + full * U; s < s0 + n; ++s) {
      float4 a[MT], b[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) b[j] = *reinterpret_cast<const float4*>(wb[j] + (size_t)s * 16);
#pragma unroll
      for (int i = 0; i < MT; ++i) a[i] = *reinterpret_cast<const float4*>(xa[i] + (size_t)s * 16);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = mfma4x4(a[i], b[j], acc[i][j]);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) part[(slot * MT * NT + i * NT + j) * 64 + lane] = acc[i][j];
  }
  __syncthreads();
  if constexpr (QR) p.Y += blockIdx.z * p.part;
  constexpr int NF = EPI == 2 ? MT * NT / 2 : MT * NT;  // (gate and up fragments finish together)
  for (int it = threadIdx.x; it < NF * 64; it += 64 * NW) {
    const int f = it >> 6, i = EPI == 2 ? f / (NT / 2) : f / NT, j = EPI == 2 ? 2 * (f % (NT / 2)) : f % NT;
    f32x4 v0 = {}, v1 = {};
#pragma unroll
    for (int q = 0; q < (QR ? 1 : 4); ++q) {
      f32x4 z0 = {}, z1 = {};
#pragma unroll
      for (int k = q * (KS / 4); k < (q + 1) * (KS / 4); ++k) {
        z0 += part[(k * MT * NT + i * NT + j) * 64 + lane];
        if constexpr (EPI == 2) z1 += part[(k * MT * NT + i * NT + j + 1) * 64 + lane];
      }
      v0 += z0;
      if constexpr (EPI == 2) v1 += z1;
    }
    store4<EPI>(p, m0 + 16 * i + 4 * g, EPI == 2 ? (n0 + 16 * j) / 2 + rl : n0 + 16 * j + rl, v0, v1);
  }
}

// Bound by the f32 MFMA (157 TFLOP/s; a large product of the library reaches 148): 110 TFLOP/s at 777 x 32768 x 1024, 103 .. 116 at
// 1024 x 2048 x 8192.
// KW groups of 4 waves (2 x 2), 16 FM x 16 FN outputs a wave; group kw multiplies 4 / KW quarters of K's 32-deep slices
// and the groups add up through LDS at the end (a second group gives every SIMD a wave to run while the other
// one waits for its operands).  A slice in LDS: A [32 FM rows][8 chunks of 16 B], then B [32 FN rows] alike, chunk c
// of row r at slot c ^ ((r >> 1) & 7) (a read's 16-lane groups hit distinct banks).  NS stages of KW slices, all but
// the one being read in flight.
// The operands are read as f32x4: HIP's float4 is a struct, whose copy says nothing of types, and in front of such a read of LDS the
// compiler waits for every LDS-DMA in flight (vmcnt(0)), the next stage's among them.  Same bits; 777 x 32768 x 1024 475 -> 429 us,
// 777 x 1024 x 6144 132 -> 115, 64 x 8720 x 1024 27.0 -> 22.8.
template <int EPI, int FM, int FN, int KW, int NS>
__global__ __launch_bounds__(256 * KW, 4) void tiles_f32_kernel(GemmF32Params p, int lr) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int BM = 32 * FM, BN = 32 * FN, SLICE = (BM + BN) * 128, STAGE = KW * SLICE;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int rl = lane & 15, g = lane >> 4, wm = w & 1, wn = w >> 1;
  const int mb = (p.M + BM - 1) / BM, tile = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = tile % mb * BM, n0 = tile / mb * BN;  // (row blocks of a column block follow one another: W from L2)
  const int slices = (p.K + 31) / 32;                                        // this group's: from beg to end, in runs r .. r1
  const int r1 = ((kw + 1) << lr) / KW;
  int r = (kw << lr) / KW;
  const int beg = slices * r >> lr, end = slices * r1 >> lr;
  // byte offsets of this lane's pieces in slice 0 (rows past the end: outside of every resource, zeros)
  constexpr unsigned kPast = 0xFFFFFFF0u;
  unsigned xo[FM], wo[FN];
  const int ch = (lane & 7) ^ (4 * (w & 1) + (lane >> 4));                   // chunk: slot ^ ((row >> 1) & 7) of row 8 (4 it + w) + lane / 8
#pragma unroll
  for (int it = 0; it < FM; ++it) {
    const int row = 8 * (it * 4 + w) + (lane >> 3);
    xo[it] = row < p.M - m0 ? ((unsigned)row * (unsigned)p.ldx + 4 * ch) * 4u : kPast;
  }
#pragma unroll
  for (int it = 0; it < FN; ++it) {
    const int row = 8 * (it * 4 + w) + (lane >> 3);
    wo[it] = row < p.N - n0 ? ((unsigned)row * (unsigned)p.K + 4 * ch) * 4u : kPast;
  }
  const size_t xb = ((size_t)(min(BM, p.M - m0) - 1) * p.ldx + p.K) * 4, wb = (size_t)min(BN, p.N - n0) * p.K * 4;
  // A slice is a scalar offset; one past the group's last reads nothing (an empty resource), and the chunks past K of a half
  // slice neither.  (With the offsets computed for every slice the runs' additions showed: 777 x 32768 x 1024 500 us, 473 so,
  // 480 without runs.)
  auto issue = [&](int s, char* buf) {
    buf += kw * SLICE;
    const bool in = beg + s < end, half = (p.K & 16) && beg + s == slices - 1;
    const int so = in ? (beg + s) * 128 : 0;
    auto piece = [&](const float* base, size_t bytes, unsigned off, int q, char* to) {
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, in ? (int)bytes : 0, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(to + q * 1024), 16,
                                               half && ch >= 4 ? kPast : off, so, 0, 0);
    };
#pragma unroll
    for (int it = 0; it < FM; ++it) piece(p.X + (size_t)m0 * p.ldx, xb, xo[it], it * 4 + w, buf);
#pragma unroll
    for (int it = 0; it < FN; ++it) piece(p.W + (size_t)n0 * p.K, wb, wo[it], it * 4 + w, buf + BM * 128);
  };
  f32x4 acc[FM][FN] = {}, run[FM][FN] = {}, sum[FM][FN] = {};  // the run's, the quarter's, KW 1: all quarters', KW 2: the first one's
  auto each = [](auto f) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) f(i, j);
  };
  const f32x4 zero = {};
  const int n = (slices + KW - 1) / KW;
  // (stages past a group's last are issued too: they read nothing, and the wait stays one constant)
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s, lds + s * STAGE);
  for (int s = 0, at = 0; s < n; ++s, at = at + 1 == NS ? 0 : at + 1) {
    const char* buf = lds + at * STAGE + kw * SLICE;
    // this stage landed everywhere, and every wave is done reading the one before, which the next issue overwrites
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * (FM + FN)) : "memory");
    issue(s + NS - 1, lds + (at == 0 ? NS - 1 : at - 1) * STAGE);
    f32x4 a[2][FM], b[2][FN];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int slot = ((4 * t + g) ^ (rl >> 1)) << 4;
#pragma unroll
      for (int i = 0; i < FM; ++i) a[t][i] = *reinterpret_cast<const f32x4*>(buf + (wm * 16 * FM + 16 * i + rl) * 128 + slot);
#pragma unroll
      for (int j = 0; j < FN; ++j) b[t][j] = *reinterpret_cast<const f32x4*>(buf + (BM + wn * 16 * FN + 16 * j + rl) * 128 + slot);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        each([&](int i, int j) {
          acc[i][j] = mfma4(a[t][i][e], b[t][j][e], acc[i][j]);
        });
    while (r < r1 && (slices * (r + 1) >> lr) <= beg + s + 1) {  // the ends of runs and quarters
      each([&](int i, int j) { run[i][j] += acc[i][j], acc[i][j] = zero; });
      if ((++r & ((1 << lr) / 4 - 1)) == 0 && (KW == 1 || (KW == 2 && r < r1)))
        each([&](int i, int j) { sum[i][j] += run[i][j], run[i][j] = zero; });
    }
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (no DMA outlives its stage)
  if constexpr (KW > 1) {
    constexpr int QN = KW == 2 ? 2 : 1, GROUP = 4 * FM * FN * 64;  // quarters of a group
    f32x4* part = reinterpret_cast<f32x4*>(lds) + w * FM * FN * 64 + lane;
    static_assert((KW - 1) * QN * GROUP * 16 <= NS * STAGE, "the other groups' quarters fit the stages");
    if (kw > 0) {
      f32x4* mine = part + (kw - 1) * QN * GROUP;
      each([&](int i, int j) {
        mine[(i * FN + j) * 64] = QN == 2 ? sum[i][j] : run[i][j];
        if constexpr (QN == 2) mine[GROUP + (i * FN + j) * 64] = run[i][j];
      });
    }
    __syncthreads();
    if (kw > 0) return;
    each([&](int i, int j) {
      sum[i][j] += run[i][j];                        // (KW 4: sum is 0)
#pragma unroll
      for (int k = 0; k < (KW - 1) * QN; ++k) sum[i][j] += part[k * GROUP + (i * FN + j) * 64];
    });
  }
  const int m = m0 + wm * 16 * FM + 4 * g, c = n0 + wn * 16 * FN;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; j += EPI == 2 ? 2 : 1)
      store4<EPI>(p, m + 16 * i, EPI == 2 ? (c + 16 * j) / 2 + rl : c + 16 * j + rl, sum[i][j], sum[i][EPI == 2 ? j + 1 : j]);
}

template <int EPI, int MT, int NT, int KS, int U, int NW = KS>
void launch_rows(const GemmF32Params& p, hipStream_t st) {
  const dim3 grid((p.N + 16 * NT - 1) / (16 * NT), (p.M + 16 * MT - 1) / (16 * MT));
  hipLaunchKernelGGL((rows_f32_kernel<EPI, MT, NT, KS, U, NW>), grid, dim3(64 * NW), 0, st, p);
}

// log2 of the runs of K: 16 where a few rows' workgroups of 16 columns leave half the CUs idle (16 waves draw more bytes than 8)
// and K is long enough for 16 steps or more to a wave, else 8.  Not of the rows or the tile: see above.  What one order costs
// against an order of each kernel's own: over 151 shapes (1 .. 1024 rows, K 1024 .. 8192) the times are 0.99, single ones up to
// 1.05 (16 x 4096 x 8192 42.2 -> 44.2 us); the error is lower (777 x 32768 x 1024: 5.7e-7 -> 2.1e-7 of the result).
template <int EPI>
int runs_log2(const GemmF32Params& p) { return EPI != 2 && p.N <= 2048 && p.K >= 4096 ? 4 : 3; }

template <int EPI, int KW>
void launch_tiles(const GemmF32Params& p, hipStream_t st) {
  constexpr int F = 2, NS = 2;
  const int tiles = ((p.M + 32 * F - 1) / (32 * F)) * ((p.N + 32 * F - 1) / (32 * F));
  hipLaunchKernelGGL((tiles_f32_kernel<EPI, F, F, KW, NS>), dim3(tiles), dim3(256 * KW), NS * KW * 64 * F * 128, st, p, runs_log2<EPI>(p));
}

int cdiv(int a, int b) { return (a + b - 1) / b; }

template <int EPI>
void launch(const GemmF32Params& p, hipStream_t st) {
  const int64_t t64 = (int64_t)cdiv(p.M, 64) * cdiv(p.N, 64);
  const bool fits = (int64_t)64 * p.ldx * 4 < 0x7FFFFFF0ll && (int64_t)64 * p.K * 4 < 0x7FFFFFF0ll;  // (32-bit offsets in a tile)
  // Tiles from where about half the CUs get one (us, rows / tiles kernel): 64 x 8720 x 1024 (137 tiles) 37 / 27, 333 x 1024
  // x 1024 (96) 24 / 23, 128 x 2048 x 2048 (64) 23 / 43.  Waves per tile so that a CU holds 16 of them (1 / 2 / 4 groups):
  // 777 x 1024 x 6144 (208 tiles) 133 / 112 / 105, 1024 x 2048 x 8192 (512) 279 / 267 / 276, 777 x 32768 x 1024 (6656) 431 /
  // 457 / 513; the kernel without LDS or k groups that this one replaced: 202 / 507 / 777.  (Three stages of one k group: 441 and,
  // 480 x 8192 x 1024, 83 against 74.)  (A 128 x 128 tile: 290 against
  // 307 at 1024 x 8192 x 2048, but 545 against 481 at 777 x 32768 x 1024.)
  if (p.M > 32 && t64 >= 120 && fits) {
    if (t64 <= 256) return launch_tiles<EPI, 4>(p, st);
    if (t64 <= 512) return launch_tiles<EPI, 2>(p, st);
    return launch_tiles<EPI, 1>(p, st);
  }
  if constexpr (EPI != 2) {
    if (runs_log2<EPI>(p) == 4) {
      if (p.M <= 16) return launch_rows<EPI, 1, 1, 16, 4>(p, st);
      // (32 rows to a workgroup while each gets a CU of its own: 48 x 1024 x 4096 23.9 us, 37.3 in blocks of 64; 100 x 2048 x 4096 45.9 / 40.4)
      if (cdiv(p.N, 16) * cdiv(p.M, 32) <= 256) return launch_rows<EPI, 2, 1, 16, 2>(p, st);
      return launch_rows<EPI, 4, 1, 16, 2, 8>(p, st);
    }
  }
  // two column tiles per workgroup where one would already give every CU four workgroups (and for gate / up pairs)
  const bool two = EPI == 2 || cdiv(p.N, 16) * cdiv(p.M, 64) >= 1024;
  if (p.M <= 16) {
    if (two) return launch_rows<EPI, 1, 2, 8, 4>(p, st);
    if constexpr (EPI != 2) return launch_rows<EPI, 1, 1, 8, 4>(p, st);
  }
  if (p.M <= 32) {
    if (two) return launch_rows<EPI, 2, 2, 8, 2>(p, st);
    if constexpr (EPI != 2) return launch_rows<EPI, 2, 1, 8, 4>(p, st);
  }
  if (two) return launch_rows<EPI, 4, 2, 8, 2>(p, st);
  if constexpr (EPI != 2) return launch_rows<EPI, 4, 1, 8, 2>(p, st);
}

}  // namespace

namespace {
int check_f32(const GemmF32Params* p) {
  if (p->M < 1 || p->N < 1 || p->K < 16 || p->K % 16 || p->ldx % 4) return -1;
  if ((reinterpret_cast<uintptr_t>(p->X) & 15) || (reinterpret_cast<uintptr_t>(p->W) & 15)) return -2;
  return 0;
}
}  // namespace

// A product's four quarters (p->part floats apart), or -7: whole, it leaves no CU without columns, or its rows are too many
extern "C" int vwa_gemm_f32_quarters(const GemmF32Params* p, int cus, int launch, hipStream_t st) {
  if (const int rc = check_f32(p)) return rc;
  if (p->M > 16 || 2 * cdiv(p->N, 16) > cus) return -7;
  if (!launch) return 0;
  const dim3 grid(cdiv(p->N, 16), 1, 4);
  if (runs_log2<0>(*p) == 4) hipLaunchKernelGGL((rows_f32_kernel<0, 1, 1, 16, 8, 4, true>), grid, dim3(256), 0, st, *p);
  else hipLaunchKernelGGL((rows_f32_kernel<0, 1, 1, 8, 8, 2, true>), grid, dim3(128), 0, st, *p);
  return (int)hipGetLastError();
}

extern "C" int vwa_gemm_f32(int epi, const GemmF32Params* p, hipStream_t st) {
  if (const int rc = check_f32(p)) return rc;
  if (epi == 1 && !p->R) return -3;
  if (epi == 6 && (!p->Y2 || p->n_split < 0 || p->n_split > p->N)) return -4;
  if (epi == 2 && p->N % 32) return -5;
  switch (epi) {
    case 0: launch<0>(*p, st); break;
    case 1: launch<1>(*p, st); break;
    case 2: launch<2>(*p, st); break;
    case 6: launch<6>(*p, st); break;
    default: return -6;
  }
  return (int)hipGetLastError();
}
