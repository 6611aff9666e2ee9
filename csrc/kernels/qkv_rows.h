// Device parts of one row's rotation and cache write (QkvCacheParams), shared by their own launch (stack_ops.hip) and the
// scores of a decode step (talk_attention.hip).
#pragma once
#include "common.h"
#include "stack_kernels.h"
#include "stack_types.h"

namespace {
using namespace vwa;

// dimension a of a pair turned by (c, s); b: its partner; hi: of the second half
VWA_DEVICE float turned(bool hi, float a, float b, float c, float s) { return hi ? a * c + b * s : a * c - b * s; }

// Part of one row.  VEC consecutive dimensions per thread (8 when the half rotation is a
// multiple of 8, else 1): a rotated chunk reads its partner chunk rot_dims / 2 away.  first: of the heads [q | k], the first
// that is taken (p.H: keys and values alone, no q_out).
template <class T, int VEC>
VWA_DEVICE void qkv_cache_row(const QkvCacheParams& p, int row, int part, int parts, int first = 0) {
  const T* x = reinterpret_cast<const T*>(p.x) + (size_t)row * p.ldx;
  const int64_t slot = p.slots[row];
  const int pos = min(max(p.positions[row], 0), p.max_pos - 1);
  const int64_t blk = slot >= 0 ? slot / p.block_size : 0;
  const int off = slot >= 0 ? (int)(slot % p.block_size) : 0;
  const int half = p.rot_dims >> 1;
  const float* cs = p.rope + (size_t)pos * p.rot_dims;
  const int cph = p.dk / VEC, nqk = (p.H + p.G) * cph;
  T* kc = reinterpret_cast<T*>(p.k) + blk * p.k_sb + (int64_t)off * p.dk;
  for (int u = first * cph + part * 256 + threadIdx.x; u < nqk; u += parts * 256) {
    const int head = u / cph, e = (u % cph) * VEC;
    const T* xh = x + head * p.dk;
    float o[VEC];
    if (e < p.rot_dims) {
      const bool hi = e >= half;
      const int i0 = hi ? e - half : e, pe = hi ? e - half : e + half;
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float a = ldv(xh + e + j), b = ldv(xh + pe + j);
        const float c = cs[2 * (i0 + j)], s = cs[2 * (i0 + j) + 1];
        o[j] = turned(hi, a, b, c, s);
      }
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) o[j] = ldv(xh + e + j);
    }
    T* dst;
    if (head < p.H) {
      dst = reinterpret_cast<T*>(p.q_out) + (size_t)row * p.ldq + head * p.dk + e;
    } else {
      if (slot < 0) continue;
      dst = kc + (int64_t)(head - p.H) * p.k_sh + e;
    }
    if constexpr (VEC == 8) {
      const float lo[4] = {o[0], o[1], o[2], o[3]}, hi4[4] = {o[4], o[5], o[6], o[7]};
      st4(dst, lo);
      st4(dst + 4, hi4);
    } else {
      stv(dst, o[0]);
    }
  }
  if (slot < 0) return;
  const T* xv = x + (p.H + p.G) * p.dk;
  T* vc = reinterpret_cast<T*>(p.v) + blk * p.v_sb + off;
  for (int u = part * 256 + threadIdx.x; u < p.G * p.dv; u += parts * 256) {
    const int g = u / p.dv, d = u % p.dv;
    vc[(int64_t)g * p.v_sh + (int64_t)d * p.block_size] = xv[u];
  }
}

// EPL dimensions e .. of a head (xh; e a multiple of EPL, rot_dims / 2 of 8), the first rot_dims of them turned by the table row
// cs (16-byte aligned), as an MFMA fragment: what the row's q_out or cache entry holds.
template <class T>
VWA_DEVICE uint4 turned_frag(const T* xh, int e, int rot_dims, const float* cs) {
  constexpr int N = 16 / sizeof(T);
  const uint4 raw = *reinterpret_cast<const uint4*>(xh + e);
  const int half = rot_dims >> 1;
  const bool rot = e < rot_dims, hi = e >= half;
  const int i0 = !rot ? 0 : hi ? e - half : e, pe = !rot ? e : hi ? e - half : e + half;
  const uint4 par = *reinterpret_cast<const uint4*>(xh + pe);
  float4 t[N / 2];
#pragma unroll
  for (int j = 0; j < N / 2; ++j) t[j] = reinterpret_cast<const float4*>(cs + 2 * i0)[j];
  float o[N];
  if constexpr (sizeof(T) == 2) {
    float a[8], b[8];
    unpack8(raw, a);
    unpack8(par, b);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = turned(hi, a[j], b[j], j & 1 ? t[j >> 1].z : t[j >> 1].x, j & 1 ? t[j >> 1].w : t[j >> 1].y);
    const uint4 y = pack8(o);
    return rot ? y : raw;
  } else {
    const float a[4] = {__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w)};
    const float b[4] = {__uint_as_float(par.x), __uint_as_float(par.y), __uint_as_float(par.z), __uint_as_float(par.w)};
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = turned(hi, a[j], b[j], j & 1 ? t[j >> 1].z : t[j >> 1].x, j & 1 ? t[j >> 1].w : t[j >> 1].y);
    const uint4 y = make_uint4(__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3]));
    return rot ? y : raw;
  }
}

}  // namespace
