// Row kernels of layer stacks with an f32 residual stream.
//
//  layernorm_f32 : y (T) = (x - mean) * rstd * w (+ b) of f32 rows, two-pass statistics in f32
//  add_norm      : x += norm(branch) * w1, h = norm(x) * w2 -- the end of a sublayer and the start of the next
//  embedding_f32 : f32 residual rows from a T table, scaled
//  qkv_cache     : partial rotation of q / k heads + paged cache write (V transposed inside a block)
//  qkv_mingru    : qkv_cache and the recurrence's rows form of a decode step in one launch
#include "mixer_kernels.h"
#include "qkv_rows.h"
#include "recurrence.h"

using namespace vwa;

namespace {

// I: a number of its own for every sum of a kernel (so one barrier each).  lds_sync: stores in flight are not waited for.
template <int I>
VWA_DEVICE float block_sum(float v, float (*red)[4]) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[I][threadIdx.x >> 6] = v;
  lds_sync();
  return (red[I][0] + red[I][1]) + (red[I][2] + red[I][3]);
}

// four weights from column c (0 past D)
VWA_DEVICE void w4(const float* w, int c, int D, float (&v)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = c + j < D ? w[min(c + j, D - 1)] : 0.f;
}

// this thread's weights of a row, STEPS x 4 as the row's columns
template <int STEPS>
VWA_DEVICE void row_weights(const float* w, int D, float (&o)[STEPS][4]) {
  const int last = (D - 1) & ~3;
  if (D % 4 == 0 && (reinterpret_cast<uintptr_t>(w) & 15) == 0) {
#pragma unroll
    for (int i = 0; i < STEPS; ++i) ld4(w + min((i * 256 + (int)threadIdx.x) * 4, last), o[i]);
  } else {
#pragma unroll
    for (int i = 0; i < STEPS; ++i) w4(w, (i * 256 + (int)threadIdx.x) * 4, D, o[i]);
  }
}

// rows k .. k + B - 1 of n, `slab` elements apart, added at this thread's columns in their order, all of their loads in flight
template <int B, int STEPS, class E>
VWA_DEVICE void add_parts(const E* b, int64_t slab, int k, int n, int last, float (&v)[STEPS][4]) {
  float u[B][STEPS][4];
#pragma unroll
  for (int e = 0; e < B; ++e)
#pragma unroll
    for (int i = 0; i < STEPS; ++i)
      ld4(b + min(k + e, n - 1) * slab + min((i * 256 + (int)threadIdx.x) * 4, last), u[e][i]);
#pragma unroll
  for (int e = 0; e < B; ++e)
#pragma unroll
    for (int i = 0; i < STEPS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] += k + e < n ? u[e][i][j] : 0.f;
}
// sum of n rows.  Another batch is another round trip to memory, a load past the last row occupies the unit: the batch by the rows left.
// us of a norm in front of a projection, three in flight -> here: 48 rows of 1024, 16 slices 4.76 -> 4.00; 1 row of 2048, 8 slices the same.
template <int STEPS>
VWA_DEVICE void sum_parts(const float* b, int64_t slab, int n, int last, float (&v)[STEPS][4]) {
#pragma unroll
  for (int i = 0; i < STEPS; ++i) ld4(b + min((i * 256 + (int)threadIdx.x) * 4, last), v[i]);
  int k = 1;
  if constexpr (STEPS == 1)
    for (; k + 7 < n; k += 15) add_parts<15>(b, slab, k, n, last, v);
  if constexpr (STEPS <= 2)
    for (; k + 3 < n; k += 7) add_parts<7>(b, slab, k, n, last, v);
  for (; k < n; k += 3) add_parts<3>(b, slab, k, n, last, v);
}

// one workgroup per row, the row held in registers: STEPS x 1024 columns, 4 per thread and step, all
// loads in flight at once (columns past the row repeat its last quad and count as zero)
constexpr int kLnSteps = 8;
// PARTS: x += the sum of `parts` rows (a projection's K slices, slab elements apart) first, in their order
template <class T, int STEPS, bool PARTS>
__global__ __launch_bounds__(256) void layernorm_f32_kernel(float* __restrict__ x, int ldx, const float* __restrict__ br, int ldb,
                                                            int64_t slab, int parts, const float* __restrict__ w,
                                                            const float* __restrict__ b, T* __restrict__ y, int ldy, int D,
                                                            int Dpad, float eps) {
  __shared__ float red[2][4];
  float* xr = x + (size_t)blockIdx.x * ldx;
  T* yr = y + (size_t)blockIdx.x * ldy;
  float v[STEPS][4], wv[STEPS][4], bv[STEPS][4];
  const int last = (D - 1) & ~3;
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const float4 f = *reinterpret_cast<const float4*>(xr + min((i * 256 + (int)threadIdx.x) * 4, last));
    v[i][0] = f.x;
    v[i][1] = f.y;
    v[i][2] = f.z;
    v[i][3] = f.w;
  }
  row_weights<STEPS>(w, D, wv);
  row_weights<STEPS>(b ? b : w, D, bv);
  if constexpr (PARTS) {
    float u[STEPS][4];
    sum_parts<STEPS>(br + (size_t)blockIdx.x * ldb, slab, parts, last, u);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int c = (i * 256 + (int)threadIdx.x) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[i][j] += u[i][j];
      if (c < D) st4(xr + c, v[i]);
    }
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int c = (i * 256 + threadIdx.x) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[i][j] = c + j < D ? v[i][j] : 0.f;
      s += v[i][j];
    }
  }
  const float mu = block_sum<0>(s, red) / (float)D;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int c = (i * 256 + threadIdx.x) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = c + j < D ? v[i][j] - mu : 0.f;
      q += d * d;
    }
  }
  const float rstd = 1.f / sqrtf(block_sum<1>(q, red) / (float)D + eps);
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int c = (i * 256 + threadIdx.x) * 4;
    if (c >= D) continue;
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = c + j < D ? (v[i][j] - mu) * rstd * wv[i][j] + (b ? bv[i][j] : 0.f) : 0.f;
    st4(yr + c, o);
  }
  for (int c = ((D + 3) & ~3) + threadIdx.x; c < Dpad; c += 256) stv(yr + c, 0.f);
}

template <class T, int STEPS>
void launch_ln_steps(float* x, int ldx, const float* br, int ldb, int64_t slab, int parts, const float* w, const float* b, T* y,
                     int ldy, int rows, int D, int Dpad, float eps, hipStream_t st) {
  if (br)
    hipLaunchKernelGGL((layernorm_f32_kernel<T, STEPS, true>), dim3(rows), dim3(256), 0, st, x, ldx, br, ldb, slab, parts, w, b, y, ldy, D, Dpad, eps);
  else
    hipLaunchKernelGGL((layernorm_f32_kernel<T, STEPS, false>), dim3(rows), dim3(256), 0, st, x, ldx, br, ldb, slab, parts, w, b, y, ldy, D, Dpad, eps);
}
template <class T>
void launch_ln(float* x, int ldx, const float* br, int ldb, int64_t slab, int parts, const float* w, const float* b, T* y, int ldy,
               int rows, int D, int Dpad, float eps, hipStream_t st) {
  if (D <= 1024) launch_ln_steps<T, 1>(x, ldx, br, ldb, slab, parts, w, b, y, ldy, rows, D, Dpad, eps, st);
  else if (D <= 2048) launch_ln_steps<T, 2>(x, ldx, br, ldb, slab, parts, w, b, y, ldy, rows, D, Dpad, eps, st);
  else if (D <= 4096) launch_ln_steps<T, 4>(x, ldx, br, ldb, slab, parts, w, b, y, ldy, rows, D, Dpad, eps, st);
  else launch_ln_steps<T, 8>(x, ldx, br, ldb, slab, parts, w, b, y, ldy, rows, D, Dpad, eps, st);
}

// mean and 1 / std of the row held as STEPS x 4 values per thread (columns past D are zero)
template <int I, int STEPS>
VWA_DEVICE float2 row_stats(const float (&v)[STEPS][4], int D, float eps, float (*red)[4]) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < STEPS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) s += v[i][j];
  const float mu = block_sum<I>(s, red) / (float)D;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < STEPS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = (i * 256 + (int)threadIdx.x) * 4 + j < D ? v[i][j] - mu : 0.f;
      q += d * d;
    }
  return make_float2(mu, 1.f / sqrtf(block_sum<I + 1>(q, red) / (float)D + eps));
}

// one workgroup per row: x += norm(sum of the branch rows) * w1; h = norm(x) * w2.  Loads of the branch,
// of the residual and of the weights are in flight together.
template <class T, int STEPS>
__global__ __launch_bounds__(256) void add_norm_kernel(float* __restrict__ x, int ldx, const T* __restrict__ br, int ldb,
                                                       int n_parts, const float* __restrict__ w1, const float* __restrict__ w2,
                                                       T* __restrict__ h, int ldh, int D, int Dpad, float eps) {
  __shared__ float red[4][4];
  float* xr = x + (size_t)blockIdx.x * ldx;
  const T* b = br + (size_t)blockIdx.x * n_parts * ldb;
  const int last = (D - 1) & ~3;
  float v[STEPS][4], xs[STEPS][4], wa[STEPS][4], wb[STEPS][4];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int c = min((i * 256 + (int)threadIdx.x) * 4, last);
    ld4(b + c, v[i]);
    ld4(xr + c, xs[i]);
  }
  row_weights<STEPS>(w1, D, wa);
  row_weights<STEPS>(w2 ? w2 : w1, D, wb);
  for (int k = 1; k < n_parts; k += 3) add_parts<3>(b, (int64_t)ldb, k, n_parts, last, v);
#pragma unroll
  for (int i = 0; i < STEPS; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if ((i * 256 + (int)threadIdx.x) * 4 + j >= D) v[i][j] = xs[i][j] = 0.f;
  const float2 sb = row_stats<0>(v, D, eps, red);
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int c = (i * 256 + threadIdx.x) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) xs[i][j] += c + j < D ? (v[i][j] - sb.x) * sb.y * wa[i][j] : 0.f;
    if (c < D) st4(xr + c, xs[i]);  // (columns past D of the last quad stay zero)
  }
  if (!w2) return;
  T* hr = h + (size_t)blockIdx.x * ldh;
  const float2 sx = row_stats<2>(xs, D, eps, red);
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    const int c = (i * 256 + threadIdx.x) * 4;
    if (c >= D) continue;
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = c + j < D ? (xs[i][j] - sx.x) * sx.y * wb[i][j] : 0.f;
    st4(hr + c, o);
  }
  for (int c = ((D + 3) & ~3) + threadIdx.x; c < Dpad; c += 256) stv(hr + c, 0.f);
}

template <class T>
void launch_add_norm(float* x, int ldx, const T* br, int ldb, int parts, const float* w1, const float* w2, T* h, int ldh,
                     int rows, int D, int Dpad, float eps, hipStream_t st) {
  const dim3 grid(rows), block(256);
  if (D <= 1024) hipLaunchKernelGGL((add_norm_kernel<T, 1>), grid, block, 0, st, x, ldx, br, ldb, parts, w1, w2, h, ldh, D, Dpad, eps);
  else if (D <= 2048) hipLaunchKernelGGL((add_norm_kernel<T, 2>), grid, block, 0, st, x, ldx, br, ldb, parts, w1, w2, h, ldh, D, Dpad, eps);
  else if (D <= 4096) hipLaunchKernelGGL((add_norm_kernel<T, 4>), grid, block, 0, st, x, ldx, br, ldb, parts, w1, w2, h, ldh, D, Dpad, eps);
  else hipLaunchKernelGGL((add_norm_kernel<T, 8>), grid, block, 0, st, x, ldx, br, ldb, parts, w1, w2, h, ldh, D, Dpad, eps);
}

template <class T>
__global__ __launch_bounds__(256) void embedding_f32_kernel(const int* __restrict__ ids, const T* __restrict__ table,
                                                            int ld, float* __restrict__ out, int ldo, int D, int Dpad,
                                                            int vocab, float scale) {
  const int row = blockIdx.x;
  const int id = ids[row];
  const bool ok = id >= 0 && id < vocab;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c < Dpad)
    out[(size_t)row * ldo + c] = ok && c < D ? ldv(table + (size_t)id * ld + c) * scale : 0.f;
}

template <class T, int VEC>
__global__ __launch_bounds__(256) void qkv_cache_kernel(QkvCacheParams p) {
  qkv_cache_row<T, VEC>(p, blockIdx.x, blockIdx.y, gridDim.y);
}

// grid.y: kQkvParts parts of the row's heads, then its recurrence channels by 256
constexpr int kQkvParts = 4;
template <class T, int VEC>
__global__ __launch_bounds__(256) void qkv_mingru_kernel(QkvCacheParams p, MinGruParams g) {
  if (blockIdx.y < kQkvParts) qkv_cache_row<T, VEC>(p, blockIdx.x, blockIdx.y, kQkvParts);
  else mingru_row<T>(g, blockIdx.x, (blockIdx.y - kQkvParts) * 256 + threadIdx.x);
}

}  // namespace

// br (optional): f32 rows [parts][rows][ldb] added to x first (x is written then)
extern "C" int vwa_layernorm_f32(float* x, int ldx, const float* br, int ldb, int parts, const float* w, const float* b, void* y,
                                 int ldy, int rows, int D, int Dpad, float eps, int f32, hipStream_t st) {
  const int q = (D + 3) & ~3;
  if (rows < 1 || D < 1 || D > kLnSteps * 1024 || Dpad < D || ldx % 4 || ldy % 4 || ldx < q || ldy < Dpad || Dpad % 4) return -1;
  if (br && (ldb % 4 || ldb < q || parts < 1)) return -2;
  const int64_t slab = (int64_t)rows * ldb;
  if (f32) launch_ln(x, ldx, br, ldb, slab, parts, w, b, reinterpret_cast<float*>(y), ldy, rows, D, Dpad, eps, st);
  else launch_ln(x, ldx, br, ldb, slab, parts, w, b, reinterpret_cast<u16*>(y), ldy, rows, D, Dpad, eps, st);
  return (int)hipGetLastError();
}

extern "C" int vwa_add_norm(float* x, int ldx, const void* br, int ldb, int n_parts, const float* w1, const float* w2, void* h,
                            int ldh, int rows, int D, int Dpad, float eps, int f32, hipStream_t st) {
  const int q = (D + 3) & ~3;
  if (rows < 1 || D < 1 || D > kLnSteps * 1024 || n_parts < 1 || ldx % 4 || ldb % 4 || ldx < q || ldb < q || !w1) return -1;
  if (w2 && (Dpad < q || Dpad % 4 || ldh % 4 || ldh < Dpad)) return -2;
  if (f32)
    launch_add_norm(x, ldx, reinterpret_cast<const float*>(br), ldb, n_parts, w1, w2, reinterpret_cast<float*>(h), ldh, rows, D,
                    Dpad, eps, st);
  else
    launch_add_norm(x, ldx, reinterpret_cast<const u16*>(br), ldb, n_parts, w1, w2, reinterpret_cast<u16*>(h), ldh, rows, D,
                    Dpad, eps, st);
  return (int)hipGetLastError();
}

extern "C" int vwa_embedding_f32(const int* ids, const void* table, int ld, float* out, int ldo, int rows, int D, int Dpad,
                                 int vocab, float scale, int f32, hipStream_t st) {
  if (rows < 1 || D < 1 || ld < D || Dpad < D || ldo < Dpad) return -1;
  if (f32)
    hipLaunchKernelGGL((embedding_f32_kernel<float>), dim3(rows, (Dpad + 255) / 256), dim3(256), 0, st, ids,
                       reinterpret_cast<const float*>(table), ld, out, ldo, D, Dpad, vocab, scale);
  else
    hipLaunchKernelGGL((embedding_f32_kernel<u16>), dim3(rows, (Dpad + 255) / 256), dim3(256), 0, st, ids,
                       reinterpret_cast<const u16*>(table), ld, out, ldo, D, Dpad, vocab, scale);
  return (int)hipGetLastError();
}

namespace {
int check_qkv(const QkvCacheParams* p) {
  return p->rows < 1 || p->H < 1 || p->G < 1 || p->dk < 1 || p->dv < 1 || p->rot_dims % 2 || p->rot_dims > p->dk ||
         p->max_pos < 1 || p->block_size < 1;
}
bool qkv_vec(const QkvCacheParams* p) {
  return (p->rot_dims / 2) % 8 == 0 && p->dk % 8 == 0 && p->ldq % 8 == 0 && p->ldx % 8 == 0 &&
         ((reinterpret_cast<uintptr_t>(p->x) | reinterpret_cast<uintptr_t>(p->rope)) & 15) == 0;  // (16-byte loads)
}
}  // namespace

extern "C" int vwa_qkv_cache(const QkvCacheParams* p, hipStream_t st) {
  if (check_qkv(p)) return -1;
  const bool vec = qkv_vec(p);
  const dim3 grid(p->rows, p->rows <= 64 ? kQkvParts : 1), block(256);
  if (p->f32) {
    if (vec) hipLaunchKernelGGL((qkv_cache_kernel<float, 8>), grid, block, 0, st, *p);
    else hipLaunchKernelGGL((qkv_cache_kernel<float, 1>), grid, block, 0, st, *p);
  } else {
    if (vec) hipLaunchKernelGGL((qkv_cache_kernel<u16, 8>), grid, block, 0, st, *p);
    else hipLaunchKernelGGL((qkv_cache_kernel<u16, 1>), grid, block, 0, st, *p);
  }
  return (int)hipGetLastError();
}

extern "C" int vwa_qkv_mingru(const QkvCacheParams* p, const MinGruParams* g, hipStream_t st) {
  if (check_qkv(p) || g->rows != p->rows || g->width < 1 || g->f32 != p->f32) return -1;
  const bool vec = qkv_vec(p);
  const dim3 grid(p->rows, kQkvParts + (g->width + 255) / 256), block(256);
  if (p->f32) {
    if (vec) hipLaunchKernelGGL((qkv_mingru_kernel<float, 8>), grid, block, 0, st, *p, *g);
    else hipLaunchKernelGGL((qkv_mingru_kernel<float, 1>), grid, block, 0, st, *p, *g);
  } else {
    if (vec) hipLaunchKernelGGL((qkv_mingru_kernel<u16, 8>), grid, block, 0, st, *p, *g);
    else hipLaunchKernelGGL((qkv_mingru_kernel<u16, 1>), grid, block, 0, st, *p, *g);
  }
  return (int)hipGetLastError();
}
