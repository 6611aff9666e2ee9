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
// Bound by its round trips (decoded rows): the first chunk's and value's projections are asked for in front of the row's ids, a chunk
// by 16-byte loads (by elements they were 32 loads), and a block size that is a power of two divides nothing.
template <class T, int VEC>
VWA_DEVICE void qkv_cache_row(const QkvCacheParams& p, int row, int part, int parts, int first = 0) {
  const T* x = reinterpret_cast<const T*>(p.x) + (size_t)row * p.ldx;
  const T* xv = x + (p.H + p.G) * p.dk;
  const int half = p.rot_dims >> 1;
  const int cph = p.dk / VEC, nqk = (p.H + p.G) * cph, nv = p.G * p.dv;
  struct Chunk {
    float a[VEC], b[VEC];  // its dimensions, their partners
  };
  auto load = [&](Chunk& c, int u) {
    const int e = u % cph * VEC, pe = e < p.rot_dims ? (e >= half ? e - half : e + half) : e;
    const T* xh = x + u / cph * p.dk;
    if constexpr (VEC == 8) {
      ld8(xh + e, c.a);
      ld8(xh + pe, c.b);
    } else {
      c.a[0] = ldv(xh + e);
      c.b[0] = ldv(xh + pe);
    }
  };
  const int u0 = first * cph + part * 256 + threadIdx.x, v0 = part * 256 + threadIdx.x;
  Chunk ck;
  load(ck, min(u0, nqk - 1));
  T val = xv[min(v0, nv - 1)];
  const int64_t slot = p.slots[row];
  const int pos = min(max(p.positions[row], 0), p.max_pos - 1);
  asm volatile("" ::: "memory");  // (all of them ahead of what waits for the ids)
  const int bs = p.block_size;
  int64_t blk = 0;
  int off = 0;
  if (slot >= 0) {
    blk = (bs & (bs - 1)) == 0 ? slot >> __builtin_ctz(bs) : slot / bs;
    off = (int)(slot - blk * bs);
  }
  const float* cs = p.rope + (size_t)pos * p.rot_dims;
  T* kc = reinterpret_cast<T*>(p.k) + blk * p.k_sb + (int64_t)off * p.dk;
  for (int u = u0; u < nqk; u += parts * 256) {
    const int head = u / cph, e = (u % cph) * VEC;
    if (u != u0) load(ck, u);
    float o[VEC];
    if (e < p.rot_dims) {
      const bool hi = e >= half;
      const int i0 = hi ? e - half : e;
      float t[2 * VEC];  // (cos, sin)
      if constexpr (VEC == 8) {
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<float4*>(t + 4 * j) = reinterpret_cast<const float4*>(cs + 2 * i0)[j];
      } else {
        t[0] = cs[2 * i0];
        t[1] = cs[2 * i0 + 1];
      }
#pragma unroll
      for (int j = 0; j < VEC; ++j) o[j] = turned(hi, ck.a[j], ck.b[j], t[2 * j], t[2 * j + 1]);
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) o[j] = ck.a[j];
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
  T* vc = reinterpret_cast<T*>(p.v) + blk * p.v_sb + off;
  for (int u = v0; u < nv; u += parts * 256) {
    const int g = u / p.dv, d = u % p.dv;
    if (u != v0) val = xv[u];
    vc[(int64_t)g * p.v_sh + (int64_t)d * bs] = val;
  }
}

// EPL dimensions e .. of a head (xh; e a multiple of EPL, rot_dims / 2 of 8), the first rot_dims of them turned by the table row
// cs (16-byte aligned), as an MFMA fragment: what the row's q_out or cache entry holds.
struct Turn {
  int i0, pe;      // first pair of the table row, first of the partner dimensions
  bool rot, hi;
};
VWA_DEVICE Turn turn_of(int e, int rot_dims) {
  const int half = rot_dims >> 1;
  Turn t;
  t.rot = e < rot_dims;
  t.hi = e >= half;
  t.i0 = !t.rot ? 0 : t.hi ? e - half : e;
  t.pe = !t.rot ? e : t.hi ? e - half : e + half;
  return t;
}
template <class T>
using Turns = float4[8 / sizeof(T)];  // (cos, sin) of a fragment's dimensions
template <class T>
VWA_DEVICE void load_turns(Turns<T>& t, const Turn& u, const float* cs) {
#pragma unroll
  for (int j = 0; j < (int)(8 / sizeof(T)); ++j) t[j] = reinterpret_cast<const float4*>(cs + 2 * u.i0)[j];
}
template <class T>
VWA_DEVICE uint4 turn_frag(const Turn& u, const uint4& raw, const uint4& par, const Turns<T>& t) {
  constexpr int N = 16 / sizeof(T);
  float o[N];
  if constexpr (sizeof(T) == 2) {
    float a[8], b[8];
    unpack8(raw, a);
    unpack8(par, b);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = turned(u.hi, a[j], b[j], j & 1 ? t[j >> 1].z : t[j >> 1].x, j & 1 ? t[j >> 1].w : t[j >> 1].y);
    const uint4 y = pack8(o);
    return u.rot ? y : raw;
  } else {
    const float a[4] = {__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z), __uint_as_float(raw.w)};
    const float b[4] = {__uint_as_float(par.x), __uint_as_float(par.y), __uint_as_float(par.z), __uint_as_float(par.w)};
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = turned(u.hi, a[j], b[j], j & 1 ? t[j >> 1].z : t[j >> 1].x, j & 1 ? t[j >> 1].w : t[j >> 1].y);
    const uint4 y = make_uint4(__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3]));
    return u.rot ? y : raw;
  }
}
template <class T>
VWA_DEVICE uint4 turned_frag(const T* xh, int e, int rot_dims, const float* cs) {
  const Turn u = turn_of(e, rot_dims);
  const uint4 raw = *reinterpret_cast<const uint4*>(xh + e), par = *reinterpret_cast<const uint4*>(xh + u.pe);
  Turns<T> t;
  load_turns<T>(t, u, cs);
  return turn_frag<T>(u, raw, par, t);
}

}  // namespace
