// Routed experts.
//
//  moe_route : sigmoid router scores (MFMA, f32 sums), the best ``top`` experts of every row, and the pairs
//              (row, choice) grouped by expert into tiles of at most ``tile`` pairs -- by the last workgroup
//  moe_gemm  : the experts' matrices over such a tile (here tiles of 16 or 32 pairs, streaming; of 128 or 256
//              go to gemm.hip's grouped launch).  First launch: the tile's rows times gate and up, scaled
//              by the pair's score ahead of the activation (w (W h) = W (w h)); second: down, one row per pair.
//              (The pairs of a row are added, in the order of its choices, by add_norm.)
// A row's results do not depend on the tile it lands in, so the order inside an expert is free.
#include "mixer_kernels.h"
#include "stack_types.h"
#include "vwa_kernels.h"

using namespace vwa;

namespace {

constexpr size_t kMaxLds = 160 * 1024 - 8192;
constexpr int kRouteWaves = 8, kRouteThreads = kRouteWaves * 64, kMaxExperts = 256;

// Experts whose places among a row's choices are counted: a lane each of the 32 that a row has.  The launch is bound by its serial
// chain (loads, sums, choices, groups), and the choices one after another are top x 5 dependent exchanges of it.  us, chosen in turn ->
// counted, top 4: bf16, K 2048, 16 rows of 16 experts 8.1 -> 6.5; K 1024, 48 rows 9.2 -> 7.5; 24 experts 10.5 -> 9.2; f32, K 1024,
// 4 rows 7.5 -> 6.0.  Of more experts than lanes a lane would count several, and a maximum after another stays; so it does where few are
// chosen of many, since the count goes over all of them: one of 32 6.5 -> 7.0 (K 256, 1 row) and 24.7 -> 25.3, one of 16 the same.
constexpr int kRankExperts = 32;
bool ranks(int E, int top) { return E <= kRankExperts && E <= 16 * top; }
// A score as it is ranked: one that is not a number is ahead of every other (they are <= 1) and its weight shows it, as torch.topk has it
constexpr float kNoNumber = 2.f;
VWA_DEVICE float rank_of(float score) { return score == score ? score : kNoNumber; }
VWA_DEVICE float weight_of(float rank) { return rank == kNoNumber ? __builtin_nanf("") : rank; }

// pairs -> tiles of one expert each (the whole workgroup); id_of(pair): its expert
// (One wave that counts expert after expert from ballots, without LDS and barriers: 0.25 us an expert.)
template <class F>
VWA_DEVICE void group_pairs(const MoeRouteParams& p, F&& id_of) {
  __shared__ int cnt[kMaxExperts], first[kMaxExperts], s_total;
  const int tid = threadIdx.x, P = p.rows * p.top;
  for (int e = tid; e < p.E; e += kRouteThreads) cnt[e] = 0;
  lds_sync();
  constexpr int B = 8;                               // ids whose loads are in flight together
  auto for_pairs = [&](auto&& fn) {
    for (int i0 = tid; i0 < P; i0 += B * kRouteThreads) {
      int e[B];
#pragma unroll
      for (int k = 0; k < B; ++k) e[k] = id_of(min(i0 + k * kRouteThreads, P - 1));
#pragma unroll
      for (int k = 0; k < B; ++k)
        if (i0 + k * kRouteThreads < P && e[k] >= 0) fn(i0 + k * kRouteThreads, e[k]);
    }
  };
  for_pairs([&](int, int e) { atomicAdd(&cnt[e], 1); });
  lds_sync();
  if (tid < 64) {                                    // exclusive prefix of the experts' tile counts
    int base = 0;
    for (int e0 = 0; e0 < p.E; e0 += 64) {
      const int e = e0 + tid, n = e < p.E ? (cnt[e] + p.tile - 1) / p.tile : 0;
      int x = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (tid >= o) x += y;
      }
      if (e < p.E) first[e] = base + x - n;
      base += __shfl(x, 63, 64);
    }
    if (tid == 0) s_total = base;
  }
  lds_sync();
  for (int e = tid; e < p.E; e += kRouteThreads) {
    const int n = cnt[e];
    for (int k = 0; k * p.tile < n; ++k) {
      int* t = p.tiles + 1 + 3 * (first[e] + k);
      t[0] = e;
      t[1] = (first[e] + k) * p.tile;
      t[2] = min(p.tile, n - k * p.tile);
    }
  }
  if (tid == 0) p.tiles[0] = s_total;
  lds_sync();
  for (int e = tid; e < p.E; e += kRouteThreads) cnt[e] = first[e] * p.tile;
  lds_sync();
  for_pairs([&](int i, int e) { p.order[atomicAdd(&cnt[e], 1)] = i; });
}

// tiles that n <= 16 pairs (a workgroup's rows) take
VWA_DEVICE int small_tiles(int n, int tile) { return tile >= 16 ? (n > 0 ? 1 : 0) : (n + tile - 1) / tile; }
// Sum over a half wave's lanes up to this one
VWA_DEVICE int half_prefix(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);  // (from 1, 2, 4, 8 lanes below within 16, zero past their end)
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
  return v + __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, true);  // (the sixteen below: their last lane's)
}

template <class T, bool COUNT>
__global__ __launch_bounds__(kRouteThreads) void moe_route_kernel(MoeRouteParams p) {
  using M = MM<T>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int s_last, s_pairs[kRankExperts];
  const int tid = threadIdx.x, lane = lane_id(), w = __builtin_amdgcn_readfirstlane(tid >> 6), rl = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.x * 16, nr = min(16, p.rows - r0), et = (p.E + 15) / 16, Ep = et * 16, steps = p.K / M::KS;
  float* red = reinterpret_cast<float*>(smem);       // [waves][Ep][16 rows]
  float* sc = red + kRouteWaves * Ep * 16;           // [16 rows][Ep + 1]
  const T* h = reinterpret_cast<const T*>(p.h) + (size_t)(r0 + min(rl, nr - 1)) * p.ldh + g * M::EPL;
  const uint4* wf = reinterpret_cast<const uint4*>(p.w) + lane;
  const bool live = p.slots[r0 + min(tid >> 5, nr - 1)] >= 0;  // (of the row whose experts this thread chooses)
  if (COUNT && tid < kRankExperts) s_pairs[tid] = 0;
  for (int e = 0; e < et; ++e) {                     // D[expert 4 g + i][row rl], every wave a part of K
    f32x4 acc = {};
    for (int s0 = w; s0 < steps; s0 += 8 * kRouteWaves) {
      uint4 a[8], b[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int s = min(s0 + u * kRouteWaves, steps - 1);
        a[u] = wf[((size_t)e * steps + s) * 64];
        b[u] = *reinterpret_cast<const uint4*>(h + s * M::KS);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (s0 + u * kRouteWaves < steps) acc = M::mma(a[u], b[u], acc);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) red[(w * Ep + e * 16 + 4 * g + i) * 16 + rl] = acc[i];
  }
  lds_sync();
  for (int i = tid; i < Ep * 16; i += kRouteThreads) {
    float z = 0.f;
#pragma unroll
    for (int k = 0; k < kRouteWaves; ++k) z += red[k * Ep * 16 + i];
    sc[(i & 15) * (Ep + 1) + (i >> 4)] = (i >> 4) < p.E ? rank_of(1.f / (1.f + expf(-z))) : -2.f;
  }
  lds_sync();
  const int r = tid >> 5, q = tid & 31, row = r0 + r;  // 32 lanes per row: the choices stay inside a wave
  if constexpr (COUNT) {
    // an expert's place is the number of experts ahead of it (a larger score; of equal ones the lower number): all choices at once
    // where one maximum after another is a chain of lane exchanges.
    const float* s = sc + r * (Ep + 1);
    const float v = s[min(q, p.E - 1)];
    int place = q < p.E ? 0 : p.E;
#pragma unroll 4
    for (int o = 0; o < p.E; ++o) {
      const float u = s[o];
      place += u > v || (u == v && o < q) ? 1 : 0;
    }
    const bool chosen = place < p.top && r < nr;
    if (gridDim.x == 1) {
      // one workgroup: the lane that has chosen an expert takes the pair's place in its group with the count, and every half wave adds up
      // the experts' tiles in front: one barrier where counting, adding up and placing the pairs one after another are five.  (us, with
      // them -> here, top 4 of 16: bf16, K 2048, 16 rows 8.3 -> 6.2; f32, K 1024, 4 rows 7.7 -> 6.3.)
      const int at = chosen && live ? atomicAdd(&s_pairs[q], 1) : 0;
      lds_sync();
      const int pairs = s_pairs[q], n = small_tiles(pairs, p.tile), first = half_prefix(n) - n;
      if (chosen) {
        const int pair = row * p.top + place;
        p.wts[pair] = live ? weight_of(v) : 0.f;
        p.ids[pair] = live ? q : -1;
        if (live) p.order[first * p.tile + at] = pair;
      }
      if (tid < 32) {
        for (int k = 0; k < n; ++k) {
          int* tl = p.tiles + 1 + 3 * (first + k);
          tl[0] = q;
          tl[1] = (first + k) * p.tile;
          tl[2] = min(p.tile, pairs - k * p.tile);
        }
        if (tid == 31) p.tiles[0] = first + n;
      }
      return;
    }
    if (chosen) {
      p.wts[row * p.top + place] = live ? weight_of(v) : 0.f;
      __hip_atomic_store(p.ids + row * p.top + place, live ? q : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  } else {
    int* lds_ids = reinterpret_cast<int*>(red);      // (a launch of one workgroup groups from here)
    for (int k = 0; k < p.top; ++k) {
      float best = -3.f;
      int at = 0;
      for (int e = q; e < p.E; e += 32) {
        const float v = sc[r * (Ep + 1) + e];
        if (v > best) {
          best = v;
          at = e;
        }
      }
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) {
        const float bo = __shfl_xor(best, o, 32);
        const int ao = __shfl_xor(at, o, 32);
        if (bo > best || (bo == best && ao < at)) {
          best = bo;
          at = ao;
        }
      }
      if (q == 0 && r < nr) {
        sc[r * (Ep + 1) + at] = -1.f;                // (taken; scores are positive)
        p.wts[row * p.top + k] = live ? weight_of(best) : 0.f;
        lds_ids[r * p.top + k] = live ? at : -1;
        __hip_atomic_store(p.ids + row * p.top + k, live ? at : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    lds_sync();
    if (gridDim.x == 1) {
      group_pairs(p, [&](int i) { return lds_ids[i]; });
      return;
    }
  }
  // ---- the last workgroup groups the pairs
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_sync();
  if (tid == 0) {
    const int t = __hip_atomic_fetch_add(p.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = t == (int)gridDim.x - 1;
    if (s_last) __hip_atomic_store(p.ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  lds_sync();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  group_pairs(p, [&](int i) { return __hip_atomic_load(p.ids + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); });
}

// ------------------------------------------------------------------------------------------ small tiles (16 NP pairs)
// A workgroup per (tile, NU x 16 features | columns); its 4 waves split K, the sums meet in LDS.  Bound by the experts' weights
// arriving: SUB substeps of a wave's k-groups (of 4 each) are requested before the products of the SUB before; SUB 0: a k-group
// is requested when the one before is done, which leaves registers for twice the workgroups (launch_small chooses).
template <class T, bool DOWN, int NP, int NU, int SUB>
__global__ __launch_bounds__(256, SUB ? 2 : 1) void moe_small_kernel(MoeGemmParams p) {
  using M = MM<T>;
  constexpr int NA = DOWN ? 1 : 2;                   // 16-row tiles of the matrix per unit
  __shared__ float red[4][NP][NU][NA][64][4];
  const int tile = blockIdx.y;
  if (tile >= p.tiles[0]) return;
  const int e = p.tiles[1 + 3 * tile], place = p.tiles[2 + 3 * tile], n = p.tiles[3 + 3 * tile];
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, g = lane >> 4;
  const int KG = p.K / (16 * M::EPL), units = p.N / (16 * NA), unit0 = blockIdx.x * NU;
  const T* x[NP];
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    const int src = place + min(16 * t + rl, n - 1);
    x[t] = reinterpret_cast<const T*>(p.x) + (size_t)(DOWN ? src : p.order[src] / p.top) * p.ldx + 4 * M::EPL * g;
  }
  const uint4* wp[NU];                               // (a unit past the matrix repeats its last one)
#pragma unroll
  for (int u = 0; u < NU; ++u)
    wp[u] = reinterpret_cast<const uint4*>(reinterpret_cast<const T*>(p.w) + e * p.w_expert) + (size_t)min(unit0 + u, units - 1) * NA * KG * 256;
  f32x4 acc[NP][NU][NA] = {};
  if constexpr (SUB == 0) {
    for (int kg = w; kg < KG; kg += 4) {
      uint4 f[NU][NA][4], a[NP][4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int j = 0; j < NA; ++j) f[u][j][s] = (wp[u] + ((size_t)j * KG + kg) * 256 + s * 64)[(unsigned)lane];
#pragma unroll
        for (int t = 0; t < NP; ++t) a[t][s] = *reinterpret_cast<const uint4*>(x[t] + kg * 16 * M::EPL + s * M::EPL);
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < NP; ++t)
#pragma unroll
          for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int j = 0; j < NA; ++j) acc[t][u][j] = M::mma(a[t][s], f[u][j][s], acc[t][u][j]);
    }
  } else {
    u32x4 f[2][NU][NA][SUB], a[2][NP][SUB];
    auto load = [&](int b, int kg, int s0) {         // substeps s0 .. of a k-group
#pragma unroll
      for (int s = 0; s < SUB; ++s) {
#pragma unroll
        for (int u = 0; u < NU; ++u)
#pragma unroll
          for (int j = 0; j < NA; ++j)
            f[b][u][j][s] = *reinterpret_cast<const u32x4*>(wp[u] + ((size_t)j * KG + kg) * 256 + (s0 + s) * 64 + (unsigned)lane);
#pragma unroll
        for (int t = 0; t < NP; ++t) a[b][t][s] = *reinterpret_cast<const u32x4*>(x[t] + kg * 16 * M::EPL + (s0 + s) * M::EPL);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](int b) {
#pragma unroll
      for (int s = 0; s < SUB; ++s)
#pragma unroll
        for (int t = 0; t < NP; ++t)
#pragma unroll
          for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int j = 0; j < NA; ++j)
              acc[t][u][j] = M::mma(__builtin_bit_cast(uint4, a[b][t][s]), __builtin_bit_cast(uint4, f[b][u][j][s]), acc[t][u][j]);
      __builtin_amdgcn_sched_barrier(0);
    };
    if (w < KG) load(0, w, 0);
    if constexpr (SUB == 2) {
      for (int kg = w; kg < KG; kg += 4) {
        load(1, kg, 2);
        products(0);
        if (kg + 4 < KG) load(0, kg + 4, 0);
        products(1);
      }
    } else {
      for (int kg = w; kg < KG; kg += 8) {
        if (kg + 4 < KG) load(1, kg + 4, 0);
        products(0);
        if (kg + 8 < KG) load(0, kg + 8, 0);
        if (kg + 4 < KG) products(1);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NP; ++t)
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int j = 0; j < NA; ++j) *reinterpret_cast<f32x4*>(red[w][t][u][j][lane]) = acc[t][u][j];
  __syncthreads();
  // thread (lane, i = wave): pairs 16 t + 4 g + i, column rl
  T* y = reinterpret_cast<T*>(p.y);
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    const int q = 16 * t + 4 * g + w;
    if (q >= n) continue;
    const int pair = p.order[place + q];
    const float score = DOWN ? 1.f : p.wts[pair];
    T* yr = y + (size_t)(DOWN ? pair : place + q) * p.ldy + unit0 * 16 + rl;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if (unit0 + u >= units) continue;
      float v[NA];
#pragma unroll
      for (int j = 0; j < NA; ++j)
        v[j] = (red[0][t][u][j][lane][w] + red[1][t][u][j][lane][w]) + (red[2][t][u][j][lane][w] + red[3][t][u][j][lane][w]);
      if constexpr (DOWN) stv(yr + u * 16, v[0]);
      else stv(yr + u * 16, silu(score * v[0]) * (score * v[1]));
    }
  }
}

// (units: as many matrix tiles per row of x read, gate / up or down)
// Two sets of whole k-groups, or, for 32-bit gate / up, of halves (120 registers or 72).  Against one set at a time, mean over 22
// to 45 shapes (widths 512 .. 4096, 1 .. 64 rows): 16-pair tiles 0.86 gate / up and 0.87 down, in 32 bits 0.89 (halves; whole: 0.905, and
// up to 1.08) and 0.86; 32-pair tiles 0.96 and 0.93, single shapes up to 1.03 (down, 3072 x 1024: 20.8 -> 21.4 us).  32-pair gate / up
// of up to four k-groups to a wave keeps one set where two would run in a second round of the CUs (240 registers: two
// workgroups a CU) and one does not (five): 48 rows of 2048 x 2048, 16 experts, 47.3 us (50.5 with two), 1024 x 2048 26.2 (27.5); but
// 13.8 (12.4) of 1024 x 1024, one round, 49.1 (49.9) of 1024 x 4096, rounds either way, and 97.9 (91.6) of 4096 x 2048.
constexpr int kCus = 256;
template <class T, int NP>
void launch_small(const MoeGemmParams& p, hipStream_t st) {
  constexpr int NG = NP, ND = NP == 1 ? 1 : 2 * NP;
  const int units = p.N / (p.down ? 16 : 32), nu = p.down ? ND : NG;
  const dim3 grid((units + nu - 1) / nu, p.max_tiles), block(256);
  const int64_t live = (int64_t)grid.x * (p.max_tiles - (int64_t)p.x_rows * p.top / p.tile);  // workgroups if no expert has a second tile
  if (p.down) hipLaunchKernelGGL((moe_small_kernel<T, true, NP, ND, 4>), grid, block, 0, st, p);
  else if constexpr (NP == 2) {
    if (p.K <= 16 * 128 && live > 2 * kCus && live <= 5 * kCus) hipLaunchKernelGGL((moe_small_kernel<T, false, NP, NG, 0>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((moe_small_kernel<T, false, NP, NG, 4>), grid, block, 0, st, p);
  } else {
    hipLaunchKernelGGL((moe_small_kernel<T, false, NP, NG, sizeof(T) == 4 ? 2 : 4>), grid, block, 0, st, p);
  }
}

}  // namespace

// Whether a row's choices are counted into their places (else: one maximum after another)
extern "C" int vwa_moe_ranks(int E, int top) { return ranks(E, top); }

extern "C" int vwa_moe_route(const MoeRouteParams* p, hipStream_t st) {
  if (p->rows < 1 || p->E < 1 || p->E > kMaxExperts || p->top < 1 || p->top > p->E || p->K % 32 || p->ldh % 8 || p->tile < 1 ||
      !p->wts || !p->ids || !p->tiles || !p->order || !p->ticket)
    return -1;
  // (every expert's last tile may be partly filled)
  const int64_t P = (int64_t)p->rows * p->top;
  if (p->max_tiles < (P < p->E ? P : p->E) + P / p->tile) return -2;
  const int Ep = (p->E + 15) / 16 * 16;
  const size_t lds = (size_t)kRouteWaves * Ep * 16 * 4 + 16 * (Ep + 1) * 4;
  if (lds > kMaxLds) return -10;
  const dim3 grid((p->rows + 15) / 16), block(kRouteThreads);
  if (ranks(p->E, p->top)) {
    if (p->f32) hipLaunchKernelGGL((moe_route_kernel<float, true>), grid, block, lds, st, *p);
    else hipLaunchKernelGGL((moe_route_kernel<u16, true>), grid, block, lds, st, *p);
  } else {
    if (p->f32) hipLaunchKernelGGL((moe_route_kernel<float, false>), grid, block, lds, st, *p);
    else hipLaunchKernelGGL((moe_route_kernel<u16, false>), grid, block, lds, st, *p);
  }
  return (int)hipGetLastError();
}

extern "C" int vwa_moe_gemm(const MoeGemmParams* p, hipStream_t st) {
  if (p->max_tiles < 1 || p->N % (p->down ? 16 : 32) || p->K % 128 || p->ldx % 8 || (p->tile != 16 && p->tile != 32 && p->tile != 128 && p->tile != 256) || !p->tiles || !p->order ||
      (!p->down && !p->wts))
    return -1;
  if ((reinterpret_cast<uintptr_t>(p->x) | reinterpret_cast<uintptr_t>(p->w)) & 15) return -2;
  if (p->tile > 32) {
    if (p->f32) return -3;
    GemmParams q{};
    q.X = reinterpret_cast<const uint16_t*>(p->x);
    q.ldx = p->ldx;
    q.W = reinterpret_cast<const uint16_t*>(p->w);
    q.w_tiled = 1;
    q.M = p->x_rows;
    q.N = p->N;
    q.K = p->K;
    q.Y = p->y;
    q.ldy = p->ldy;
    q.rstd = p->down ? nullptr : p->wts;
    q.g_tiles = p->tiles;
    q.g_order = p->order;
    q.g_max = p->max_tiles;
    q.g_tile = p->tile;
    q.g_top = p->top;
    q.g_down = p->down;
    q.g_wstride = p->w_expert;
    return vwa_gemm_grouped(p->down ? 0 : 2, &q, st);
  }
  if (p->f32) p->tile == 16 ? launch_small<float, 1>(*p, st) : launch_small<float, 2>(*p, st);
  else p->tile == 16 ? launch_small<u16, 1>(*p, st) : launch_small<u16, 2>(*p, st);
  return (int)hipGetLastError();
}
