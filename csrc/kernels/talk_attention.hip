// Windowed attention with kept first keys, mixed ("talking") heads and per-head output gates.
//
// Row i sees key j when j <= i and (i - j < window or j < keep).  With softmax weights w_g of query
// head g, head h applies sum_g talk[h][g] w_g to the values of its own kv head, so the weights of ALL
// heads for a key have to be normalised before any value is read: every form below computes the
// softmax statistics first and forms the (already normalised) mixed weights in a second pass.  The
// weights, their mixing and the statistics are f32; the mixed weights enter the value product as T.
//
// Keys are walked in 16-key tiles inside cache blocks.  The visible tiles of a row are those of the
// kept first keys, then those of the window (vis_tiles); edges are masked per key.
//
//  1) rows form (decode; any T, any sizes): launch A -- a workgroup per (row or few rows of a run, kv head, chunk of tiles)
//     computes S^T = K.Q^T on the MFMA (the kv head's query heads are the 16 columns), stores the
//     scores and the chunk's (max, sum) per head; launch B -- same grid -- folds the chunk statistics
//     of every head, mixes the chunk's weights into LDS in B-operand order and multiplies by V^T,
//     which the cache stores transposed (its A operand, no staging).  Chunks of a row are added in
//     chunk order by the last-arriving workgroup (sc1 hand-off + ticket, as decode attention).
//  2) prefill form (bf16), per 16 consecutive queries: launch A reduces the scores to log-sum-exps;
//     launch B recomputes them (a wave per few heads), mixes the heads on the MFMA and multiplies by V^T,
//     the weights passing between the waves through LDS in B-operand order.
#include "common.h"
#include "mq_attention.h"
#include "qkv_rows.h"
#include "recurrence.h"
#include "stack_kernels.h"
#include "stack_types.h"

#include <type_traits>

using namespace vwa;

namespace {

constexpr int kTile = 16;                  // keys per tile
constexpr float kLog2e = 1.4426950408889634f;

struct Vis {
  int sink, first, n;                      // kept tiles 0 .. sink-1, then tiles first ..; n in all
};
// tiles seen by queries at positions p0 .. p1 together
VWA_DEVICE Vis vis_tiles(int p0, int p1, int window, int keep) {
  Vis v;
  v.first = window > 0 ? max(0, p0 - window + 1) / kTile : 0;
  v.sink = keep > 0 ? min((keep + kTile - 1) / kTile, v.first) : 0;
  v.n = v.sink + p1 / kTile - v.first + 1;
  return v;
}
VWA_DEVICE int tile_of(const Vis& v, int t) { return t < v.sink ? t : v.first + t - v.sink; }
VWA_DEVICE bool sees(int i, int j, int window, int keep) {
  return j <= i && (window <= 0 || i - j < window || j < keep);
}

VWA_DEVICE void st_sc1_x4(__amdgpu_buffer_rsrc_t r, int off, const f32x4& v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 16);
}
VWA_DEVICE f32x4 ld_sc1_x4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16));
}

// ------------------------------------------------------------------------------------------ rows form
// A workgroup takes a unit of rows and a kv head: one row (its query heads are columns of the MFMA; decoded tokens) or
// GRP: up to p.nq = 16 / R consecutive rows of a sequence (columns: row, query head), so that a key is read and multiplied
// once for all of them.  777 rows of a 32-bit prompt, 8 / 4 heads of 128: both launches 332 -> 86 us per layer.
//
// Few rows are bound by the dependent round trips through memory (about 0.8 us each), not by bytes: everything whose address
// is known is requested first; scores are spread by a tile per wave (kTalkStat tiles a workgroup); and a mixing chunk holds CT
// = 16 tiles, so that contexts of up to 256 keys take no partial sums, tickets and merging.  1 row of 225 keys, 16 / 4 heads
// of 128: scores 5.4 -> 4.8, mixing 9.9 -> 8.4 us; 48 rows of 90 .. 250 keys, 8 / 4 heads: 7.4 -> 6.7, 10.5 -> 8.2.
// What is requested first has to be read off the assembly: a gate's sigmoid behind its load, a load in a branch, a scalar load behind
// an early return each waited for everything in front of them, and a cache place a value tile made the values wait for one another.  With
// those out, the heads' weights mixed in batches and divisions by reciprocals: mixing 8.3 -> 6.2 us (1 row), 8.05 -> 6.75 (48 rows).
constexpr int kWaves = 8;                      // of the mixing
// (CT, most tiles of a chunk: talk_chunk_tiles)

struct Chunks {
  int per, n;
};
// the visible tiles are dealt evenly to the fewest chunks; chunk c holds tiles c * per ..
template <int CT>
VWA_DEVICE Chunks chunks_of(int tiles) {
  const int k = (tiles + CT - 1) / CT, per = small_div(tiles + k - 1, k);
  return Chunks{per, small_div(tiles + per - 1, per)};
}

struct Unit {
  int row, cnt;    // first row, rows
  bool live;       // false: an inert row of a padded step
  int pos, seq;
  Vis v;
};
template <bool GRP>
VWA_DEVICE Unit unit_of(const TalkAttnParams& p, int ri) {
  Unit u;
  u.row = GRP ? p.groups[2 * ri] : p.row_list ? p.row_list[ri] : ri;
  u.cnt = GRP ? p.groups[2 * ri + 1] : 1;
  // (requested together, as vector loads: of scalar ones the compiler puts the last two behind the caller's return for inert rows)
  int row = u.row;
  asm volatile("" : "+v"(row));
  const int64_t slot = p.slots[row];
  const int pos = p.positions[row], seq = p.seq_ids[row];
  asm volatile("" ::: "memory");
  u.pos = __builtin_amdgcn_readfirstlane(pos);
  u.seq = __builtin_amdgcn_readfirstlane(seq);
  u.live = GRP || __builtin_amdgcn_readfirstlane((int)(slot >> 32)) >= 0;
  u.v = vis_tiles(u.pos, u.pos + u.cnt - 1, p.window, p.keep);
  u.v.n = min(u.v.n, p.nst * kTalkStat);  // (a position past the context that the scratch is sized for stays inside of it)
  return u;
}

// Steps of the head dimension whose operands are requested together: 128 dimensions.  (A loop over them unrolled eight times ran
// the four of bf16 one after another, in its remainder.)
template <class T>
constexpr int kScoreStep = 128 / MM<T>::KS;

// A workgroup's scores of its wave's tiles, masked, and their statistics over the workgroup
template <bool GRP, int NU>
VWA_DEVICE void store_scores(const TalkAttnParams& p, const Unit& un, int ri, int qi, int h, bool col, int chunk, const int (&key0)[NU],
                             const bool (&ok)[NU], f32x4 (&acc)[NU], float (&sm)[4][16][2]) {
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, b = lane >> 4;
  // lane (column rl, keys 4b .. 4b+3 of its tiles): mask, store, chunk statistics
  float mx = -INFINITY;
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool vis = ok[u] && sees(un.pos + qi, key0[u] + 4 * b + i, p.window, p.keep);
      acc[u][i] = vis ? acc[u][i] * p.scale : -INFINITY;
      mx = fmaxf(mx, acc[u][i]);
    }
  const size_t srow = (size_t)ri * p.nq + qi;         // scratch row
  if (col) {
#pragma unroll
    for (int u = 0; u < NU; ++u)
      if (ok[u])
        *reinterpret_cast<float4*>(p.s + (srow * p.H + h) * p.nst * (kTalkStat * kTile) +
                                   (chunk * kTalkStat + w + 4 * u) * kTile + 4 * b) =
            make_float4(acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
  }
  mx = groups_max(mx);
  float l = 0.f;
#pragma unroll
  for (int u = 0; u < NU; ++u)
#pragma unroll
    for (int i = 0; i < 4; ++i) l += acc[u][i] == -INFINITY ? 0.f : __expf(acc[u][i] - mx);
  l = groups_sum(l);
  if (b == 0) {
    sm[w][rl][0] = mx;
    sm[w][rl][1] = l;
  }
  lds_sync();
  if (threadIdx.x < 16 && col) {                       // (thread = column: its qi and r)
    float m = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) m = fmaxf(m, sm[i][rl][0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) sum += sm[i][rl][1] > 0.f ? sm[i][rl][1] * __expf(sm[i][rl][0] - m) : 0.f;
    float* st = p.stat + ((srow * p.H + h) * p.nst + chunk) * 2;
    st[0] = m;
    st[1] = sum;
  }
}

template <class T, bool GRP>
__global__ __launch_bounds__(256) void talk_scores_kernel(TalkAttnParams p) {
  using M = MM<T>;
  constexpr int NU = kTalkStat / 4;                  // tiles per wave
  __shared__ float sm[4][16][2];
  const int ri = blockIdx.x / p.G, c = blockIdx.x % p.G, chunk = blockIdx.y, r0 = blockIdx.z * 16;
  const Unit un = unit_of<GRP>(p, ri);
  if (!un.live) return;
  const Vis v = un.v;
  if (chunk * kTalkStat >= v.n) return;
  const int R = p.H / p.G, Rb = min(16, R - r0);
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, b = lane >> 4;
  const int qi = GRP ? rl / R : 0, r = GRP ? rl % R : rl;  // this column's row of the unit and query head
  const bool col = qi < un.cnt && r < Rb;
  const T* q = reinterpret_cast<const T*>(p.q) + (size_t)(un.row + min(qi, un.cnt - 1)) * p.ldq +
               (size_t)(c * R + r0 + min(r, Rb - 1)) * p.dk + b * M::EPL;
  const int lb = __builtin_ctz(p.block_size);
  const T* kp[NU];
  int key0[NU];
  bool ok[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int t = chunk * kTalkStat + w + 4 * u;
    ok[u] = t < v.n;
    key0[u] = tile_of(v, ok[u] ? t : v.n - 1) * kTile;
    const int64_t blk = p.block_table[(int64_t)un.seq * p.table_stride + (key0[u] >> lb)];
    kp[u] = reinterpret_cast<const T*>(p.k) + blk * p.k_sb + (int64_t)c * p.k_sh +
            (int64_t)((key0[u] & (p.block_size - 1)) + rl) * p.dk + b * M::EPL;
  }
  f32x4 acc[NU] = {};
  constexpr int NB = kScoreStep<T>;
  for (int k0 = 0; k0 < p.dk; k0 += NB * M::KS) {
    uint4 qf[NB], kf[NU][NB];
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      const int k = min(k0 + s * M::KS, p.dk - M::KS);
      qf[s] = *reinterpret_cast<const uint4*>(q + k);
#pragma unroll
      for (int u = 0; u < NU; ++u) kf[u][s] = *reinterpret_cast<const uint4*>(kp[u] + k);
    }
#pragma unroll
    for (int s = 0; s < NB; ++s)
      if (k0 + s * M::KS < p.dk) {
#pragma unroll
        for (int u = 0; u < NU; ++u) acc[u] = M::mma(kf[u][s], qf[s], acc[u]);
      }
  }
  store_scores<GRP, NU>(p, un, ri, qi, c * R + r0 + r, col, chunk, key0, ok, acc, sm);
}

// ---- a decode step's scores behind nothing but its projections
// What qkv_mingru does ahead of the scores (heads turned, keys and values into the cache, the recurrence) in the scores' launch: a
// launch of round trips less per layer.  The scoring workgroups turn their query themselves, and of the keys that belong to this
// step's rows of their sequence -- those other workgroups of the launch are writing to the cache -- they turn the projections; every
// other key comes from the cache.  The first workgroups write the cache and run the recurrence.
// us, both launches -> this one: 1 row of 225 keys, 16 / 4 heads of 128 and 2048 channels 9.4 -> 5.9; 48 rows of 90 .. 250 keys, 8 / 4
// heads and 1024 channels 10.9 -> 8.6.  The row's query and own key are turned once a workgroup, through LDS: every wave for itself
// took 6.6 and 10.7 (94 registers, and the table's row four times).  Bound by its round trips: ids with the row's own projections, the
// tile's place with the table's row, keys.  (The keys used to be requested behind the turned query: 5.9 -> 4.8 and 8.6 -> 7.5 us, with
// the cache's and the recurrence's workgroups down to three trips.)
constexpr int kStepParts = 2;                        // workgroups of a row's keys and values
// Scoring workgroups that a launch aims at, in whole ones to a row, kv head and 16 of its query heads, but three of them at least, which
// share the row's chunks (64 rows of 16 kv heads: 3072; none waits for another).  768 is what was resident at once beside the others while
// five workgroups fitted a CU.  The requests ahead of the first wait take registers: four fit in 16 bits (127), 1024 with the others, three
// in 32 bits (137), 768 with them.  The figures below are of five a CU; the number was not measured again.
// One a chunk of the longest context would be mostly workgroups without keys: 48 rows of 2048 tokens' room and 90 .. 250 keys, 3840
// workgroups 11.1 us, 768 10.7; 240 steps (1 .. 64 rows, 20 .. 2000 keys, six head shapes) against three launches: 0.93 of the time, and
// 0.914 so.  With one a row and kv head where they are many, a row's chunks were one after another: 64 rows x 8 kv heads of 2000 keys 111 ->
// 141 us, now 116 (16 bits: 64 rows and 1000 keys and more stay 2 - 8 % slower than three launches, and 3 - 14 % faster up to 225).
constexpr int kStepWgs = 768, kStepLeast = 3;
int step_wgs(int n, int chunks) {
  const int per = kStepWgs / n > kStepLeast ? kStepWgs / n : kStepLeast;
  return chunks < per ? chunks : per;
}

template <class T>
__global__ __launch_bounds__(256, sizeof(T) == 2 ? 4 : 3) void talk_step_kernel(TalkAttnParams p, QkvCacheParams qc, MinGruParams g, int per_row) {
  using M = MM<T>;
  static_assert(kTalkStat == 4, "a tile per wave");
  constexpr int NB = kScoreStep<T>;
  __shared__ float sm[4][16][2];
  __shared__ uint4 qs[NB][64], ks[NB][4];            // the query's fragments; those of the row's own key
  const int parts = kStepParts + (g.width + 255) / 256, n_parts = parts * p.rows;
  if ((int)blockIdx.x < n_parts) {
    const int row = small_div(blockIdx.x, parts), part = blockIdx.x - row * parts;
    if (part < kStepParts) qkv_cache_row<T, 8>(qc, row, part, kStepParts, p.H);
    else mingru_row<T>(g, row, (part - kStepParts) * 256 + threadIdx.x);
    return;
  }
  const int R = small_div(p.H, p.G), nz = (R + 15) / 16, bid = blockIdx.x - n_parts;
  const int cz = small_div(bid, p.rows * p.G), rg = bid - cz * (p.rows * p.G);
  const int ri = small_div(rg, p.G), c = rg - ri * p.G, chunk0 = small_div(cz, nz), r0 = (cz - chunk0 * nz) * 16;
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, b = lane >> 4;
  // the step's rows, one a lane: this row's place, and the first row of its run (rows of one sequence, at consecutive positions)
  const int lr = min(lane, p.rows - 1);
  const int64_t slot_l = p.slots[lr];
  const int pos_l = p.positions[lr], seq_l = p.seq_ids[lr];
  // requested with them: this wave's fragments of the query and of the row's own key, with their partners
  constexpr int SN = (NB + 3) / 4;
  const int Rb = min(16, R - r0), e0 = b * M::EPL;
  const T* x = reinterpret_cast<const T*>(qc.x);
  const T* xq = x + (size_t)ri * qc.ldx + (size_t)(c * R + r0 + min(rl, Rb - 1)) * p.dk;
  const T* xk = x + (size_t)ri * qc.ldx + (size_t)(p.H + c) * p.dk;
  uint4 fq[SN][2], fk[SN][2];
  auto load_own = [&](int k0) {
#pragma unroll
    for (int i = 0; i < SN; ++i) {
      const int e = min(k0 + (w + 4 * i) * M::KS, p.dk - M::KS) + e0, pe = turn_of(e, qc.rot_dims).pe;
      fq[i][0] = *reinterpret_cast<const uint4*>(xq + e);
      fq[i][1] = *reinterpret_cast<const uint4*>(xq + pe);
      fk[i][0] = *reinterpret_cast<const uint4*>(xk + e);
      fk[i][1] = *reinterpret_cast<const uint4*>(xk + pe);
    }
  };
  load_own(0);
  asm volatile("" ::: "memory");  // (not behind the wait for the ids)
  const int before = __shfl_up(seq_l, 1, 64), inert = __shfl_up((int)(slot_l < 0), 1, 64);
  const unsigned long long heads = __ballot(lane == 0 || before != seq_l || inert);
  if (!((__ballot(slot_l >= 0) >> ri) & 1)) return;
  const int head = 63 - __builtin_clzll(heads & ((2ull << ri) - 1ull));
  Unit un;
  un.row = ri;
  un.cnt = 1;
  un.live = true;
  un.pos = __builtin_amdgcn_readlane(pos_l, ri);
  un.seq = __builtin_amdgcn_readlane(seq_l, ri);
  un.v = vis_tiles(un.pos, un.pos, p.window, p.keep);
  un.v.n = min(un.v.n, p.nst * kTalkStat);
  const Vis v = un.v;
  const int fresh = __builtin_amdgcn_readlane(pos_l, head);  // keys fresh .. un.pos are rows head .. ri
  auto table_row = [&](int pos) { return qc.rope + (size_t)min(max(pos, 0), qc.max_pos - 1) * qc.rot_dims; };
  const float* cq = table_row(un.pos);
  const int lb = __builtin_ctz(p.block_size);
  // the scores of one chunk; First: this workgroup's first, for which the fragments asked for above are turned
  auto chunk_scores = [&](auto First, int chunk) {
    constexpr bool first = decltype(First)::value;
    const int t = chunk * kTalkStat + w;
    const bool ok[1] = {t < v.n};
    const int key0[1] = {tile_of(v, ok[0] ? t : v.n - 1) * kTile}, key = key0[0] + rl;
    const int blk = p.block_table[(int64_t)un.seq * p.table_stride + (key0[0] >> lb)];
    f32x4 acc[1] = {};
    auto part = [&](auto Own, int k0) {                  // Own: with the query and the own key in LDS (dimensions k0 ..)
      Turns<T> turns[SN];
      if constexpr (decltype(Own)::value) {
#pragma unroll
        for (int i = 0; i < SN; ++i) load_turns<T>(turns[i], turn_of(min(k0 + (w + 4 * i) * M::KS, p.dk - M::KS) + e0, qc.rot_dims), cq);
        asm volatile("" ::: "memory");                   // (not behind the wait for the tile's place)
      }
      auto turn_own = [&]() {
        if constexpr (decltype(Own)::value) {
#pragma unroll
          for (int i = 0; i < SN; ++i) {
            const int s = w + 4 * i;
            if (s >= NB || k0 + s * M::KS >= p.dk) break;
            const Turn u = turn_of(k0 + s * M::KS + e0, qc.rot_dims);
            qs[s][lane] = turn_frag<T>(u, fq[i][0], fq[i][1], turns[i]);
            ks[s][b] = turn_frag<T>(u, fk[i][0], fk[i][1], turns[i]);  // (the same of 16 lanes)
          }
          lds_sync();
        }
      };
      const T* kp = reinterpret_cast<const T*>(p.k) + (int64_t)blk * p.k_sb + (int64_t)c * p.k_sh +
                    (int64_t)((key0[0] & (p.block_size - 1)) + rl) * p.dk + e0;
      auto product = [&](const uint4& cached, int s) {
        const uint4 own = ks[s][b];
        acc[0] = M::mma(key == un.pos ? own : cached, qs[s][lane], acc[0]);
      };
      if (key0[0] + kTile <= fresh || fresh == un.pos) {
        uint4 kf[NB];
#pragma unroll
        for (int s = 0; s < NB; ++s) kf[s] = *reinterpret_cast<const uint4*>(kp + min(k0 + s * M::KS, p.dk - M::KS));
        turn_own();
#pragma unroll
        for (int s = 0; s < NB; ++s)
          if (k0 + s * M::KS < p.dk) product(kf[s], s);
      } else {                                           // keys of the run's rows in front of this one
        const bool mine = key >= fresh && key < un.pos;  // (keys past the row's are masked)
        const T* xr = x + (size_t)(mine ? head + key - fresh : ri) * qc.ldx + (size_t)(p.H + c) * p.dk;
        const float* ck = table_row(mine ? key : un.pos);
        turn_own();
#pragma unroll 1
        for (int s = 0; s < NB && k0 + s * M::KS < p.dk; ++s) {
          const uint4 old = *reinterpret_cast<const uint4*>(kp + k0 + s * M::KS), now = turned_frag(xr, k0 + s * M::KS + e0, qc.rot_dims, ck);
          product(mine ? now : old, s);
        }
      }
    };
    if constexpr (first) part(std::true_type{}, 0);
    for (int k0 = first ? NB * M::KS : 0; k0 < p.dk; k0 += NB * M::KS) {
      if (p.dk <= NB * M::KS) {                          // (as the first chunk left them)
        part(std::false_type{}, k0);
      } else {
        lds_sync();                                      // (the fragments before are read)
        load_own(k0);
        part(std::true_type{}, k0);
      }
    }
    store_scores<false, 1>(p, un, ri, 0, c * R + r0 + rl, rl < Rb, chunk, key0, ok, acc, sm);
  };
  int chunk = chunk0;
  if (chunk * kTalkStat >= v.n) return;
  chunk_scores(std::true_type{}, chunk);
  for (chunk += per_row; chunk * kTalkStat < v.n; chunk += per_row) {
    lds_sync();                                          // (the statistics' LDS is written again)
    chunk_scores(std::false_type{}, chunk);
  }
}

VWA_DEVICE float gate_of(const TalkAttnParams& p, float g) { return p.gate ? p.out_scale / (1.f + __expf(-g)) : p.out_scale; }
template <class T>
VWA_DEVICE const T* gate_at(const TalkAttnParams& p, int row, int h) { return reinterpret_cast<const T*>(p.gate) + (size_t)row * p.ldg + h; }

// LDS: mixed weights [keys / KS][64][16 B], weights [rows of the unit x heads][keys] f32, statistics [rows x heads][2]
template <class T, int CT>
size_t mix_lds(int H, int nq) {
  constexpr int CH = CT * kTile;
  return (size_t)nq * H * (2 + CH) * 4 + CH * 16 * sizeof(T);
}

template <class T, int CT, bool GRP>
__global__ __launch_bounds__(64 * kWaves) void talk_mix_kernel(TalkAttnParams p) {
  using M = MM<T>;
  constexpr int CH = CT * kTile, NT = 64 * kWaves;
  constexpr int HP = NT / CH;                        // (row, head)s side by side over the threads
  static_assert(CH % 64 == 0 && HP >= 1);
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int s_last;
  const int ri = blockIdx.x / (unsigned)p.G, c = blockIdx.x - ri * p.G, chunk = blockIdx.y, r0 = blockIdx.z * 16;
  // (all of the parameters in one round trip)
  asm volatile("" ::"s"(p.window), "s"(p.keep), "s"(p.nst), "s"(p.nch), "s"(p.talk), "s"(p.gate), "s"(p.q), "s"(p.v), "s"(p.v_sb), "s"(p.v_sh),
               "s"(p.block_table), "s"(p.table_stride), "s"(p.block_size), "s"(p.s), "s"(p.stat), "s"(p.dv), "s"(p.out), "s"(p.ldo), "s"(p.nq));
  const Unit un = unit_of<GRP>(p, ri);
  const int R = small_div(p.H, p.G), Rb = min(16, R - r0), h0 = c * R + r0;
  T* out = reinterpret_cast<T*>(p.out) + (size_t)un.row * p.ldo;
  if (!un.live) {
    if (chunk == 0)
      for (int i = threadIdx.x; i < Rb * p.dv; i += NT) stv(out + (size_t)h0 * p.dv + i, 0.f);
    return;
  }
  const Vis v = un.v;
  const Chunks ck = chunks_of<CT>(v.n);
  if (chunk >= ck.n) return;
  const int nstat = (v.n + kTalkStat - 1) / kTalkStat;                  // statistics of a (row, head)
  const int nact = ck.n, t0 = chunk * ck.per, nt = min(ck.per, v.n - t0), nkey = nt * kTile;
  const int g0 = p.talk ? 0 : h0, hn = p.talk ? p.H : Rb;               // heads whose weights are needed
  const int nw = un.cnt * hn, ncol = un.cnt * Rb;
  T* pf = reinterpret_cast<T*>(smem);                                   // mixed weights, B-operand order
  float* wt = reinterpret_cast<float*>(smem + CH * 16 * sizeof(T));     // [row][head][keys]
  float* hm = wt + nw * CH;                                             // [row][head] max
  float* hl = hm + nw;                                                  // [row][head] 1 / sum
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, b = lane >> 4;
  // ---- everything that is read is requested first, and nothing of it is waited for until all of it is on its way: the cache places
  // of the chunk's tiles (a lane each), the scores of this thread's (key; row, head)s, the mixing rows of this wave's columns, the gates,
  // the chunk statistics, and behind the places the first value tiles of this wave (16-column tiles w, w + 8, ...)
  const int lb = __builtin_ctz(p.block_size);
  const int my_key = tile_of(v, t0 + min(lane & (CT - 1), nt - 1)) * kTile;
  const int my_blk = p.block_table[(int64_t)un.seq * p.table_stride + (my_key >> lb)];
  constexpr int kPre = GRP ? 16 : 8;
  const int j = threadIdx.x & (CH - 1), hp = w / (CH / 64);             // key, first (row, head)
  const size_t srow = (size_t)ri * p.nq;
  const int64_t sld = (int64_t)p.nst * (kTalkStat * kTile);
  const float* sbase = p.s + (srow * p.H + g0) * sld + t0 * kTile + j;  // (keys past the chunk's: inside of the scratch, never used)
  auto head_of = [&](int i) { return GRP ? (i / hn) * p.H + i % hn : i; };  // (row, needed head) i from the unit's first
  auto score = [&](int i) -> const float* { return sbase + (int64_t)head_of(i) * sld; };
  float sv[kPre];
#pragma unroll
  for (int k = 0; k < kPre; ++k) sv[k] = *score(min(hp + HP * k, nw - 1));
  constexpr int kCols = 16 / HP;                                        // columns of a wave
  const bool in_lanes = p.talk && p.H <= 64;                            // lane g holds the weight of head g
  float tk[kCols];
  if (in_lanes) {
#pragma unroll
    for (int i = 0; i < kCols; ++i)
      tk[i] = p.talk[(size_t)(h0 + (GRP ? min(hp + HP * i, ncol - 1) % Rb : min(hp + HP * i, Rb - 1))) * p.H + min(lane, p.H - 1)];
  }
  const int qi = GRP ? rl / R : 0, r = GRP ? rl % R : rl;               // this column's row and query head
  const bool col = qi < un.cnt && r < Rb;
  // (an inert row of a group is zero whatever its query and its key hold)
  const bool on = !GRP || (col && p.slots[un.row + qi] >= 0);
  const T gate_raw = *(p.gate ? gate_at<T>(p, un.row + min(qi, un.cnt - 1), h0 + min(r, Rb - 1)) : reinterpret_cast<const T*>(p.q));
  auto stat = [&](int i, int k) { return *reinterpret_cast<const float2*>(p.stat + ((srow * p.H + g0 + head_of(i)) * p.nst + k) * 2); };
  const int si = threadIdx.x >> 4, sk = threadIdx.x & 15;               // this thread's first statistics
  const float2 stat0 = stat(min(si, nw - 1), min(sk, nstat - 1));
  constexpr int TPS = M::KS / kTile;                 // tiles per step (bf16 2, f32 1)
  constexpr int NST = CT / TPS;
  // place of the lane's tile (lanes past the chunk's tiles: of its last)
  const int64_t my_place = (int64_t)my_blk * p.v_sb + (int64_t)c * p.v_sh + (my_key & (p.block_size - 1));
  // (what has been asked for so far arrives with the places: behind the value loads, whose number depends on the chunk, the compiler
  // would wait for all of them)
  asm volatile("" ::"v"(stat0.x), "v"(stat0.y));
  const T* vb[NST];
#pragma unroll
  for (int s = 0; s < NST; ++s) {
    auto part = [&](int v) {
      const unsigned lo = __builtin_amdgcn_readlane(v, s * TPS), hi = __builtin_amdgcn_readlane(v, s * TPS + TPS - 1);
      return TPS == 2 && b >> 1 ? hi : lo;
    };
    const unsigned lo = part((int)my_place), hi = part((int)(my_place >> 32));
    vb[s] = reinterpret_cast<const T*>(p.v) + (int64_t)((uint64_t)hi << 32 | lo) + (int64_t)rl * p.block_size +
            (TPS == 2 ? (b & 1) : b) * M::EPL;
  }
  uint4 va[NST];
  auto load_v = [&](int d) {
#pragma unroll
    for (int s = 0; s < NST; ++s)
      if (s * TPS < nt) va[s] = *reinterpret_cast<const uint4*>(vb[s] + (int64_t)min(d, p.dv - 16) * p.block_size);
  };
  load_v(w * 16);
  // ---- statistics of every needed (row, head): 16 lanes each
  {
    struct Stat {
      float m, s;
    };
    auto add = [](Stat& a, float m, float s) {
      const float mn = fmaxf(a.m, m);
      if (s > 0.f) a.s = (a.s > 0.f ? a.s * __expf(a.m - mn) : 0.f) + s * __expf(m - mn);
      a.m = mn;
    };
    auto merge = [](Stat& a, float mo, float so) {
      const float mn = fmaxf(a.m, mo);
      a.s = (a.s > 0.f ? a.s * __expf(a.m - mn) : 0.f) + (so > 0.f ? so * __expf(mo - mn) : 0.f);
      a.m = mn;
    };
    auto finish = [&](Stat& a, int i) {
      merge(a, row_ror<8>(a.m), row_ror<8>(a.s));
      merge(a, row_ror<4>(a.m), row_ror<4>(a.s));
      merge(a, row_ror<2>(a.m), row_ror<2>(a.s));
      merge(a, row_ror<1>(a.m), row_ror<1>(a.s));
      if (sk == 0) {
        hm[i] = a.m;
        hl[i] = 1.f / a.s;
      }
    };
    Stat a{-INFINITY, 0.f};
    if (sk < nstat) add(a, stat0.x, stat0.y);
    for (int k = sk + 16; k < nstat; k += 16) {
      const float2 ms = stat(min(si, nw - 1), k);
      add(a, ms.x, ms.y);
    }
    if (si < nw) finish(a, si);
    for (int i = si + NT / 16; i < nw; i += NT / 16) {
      a = Stat{-INFINITY, 0.f};
      for (int k = sk; k < nstat; k += 16) {
        const float2 ms = stat(i, k);
        add(a, ms.x, ms.y);
      }
      finish(a, i);
    }
  }
  lds_sync();
  // ---- normalised weights of the chunk's keys (0 past the last tile)
  auto weight = [&](float s, float m, float l) {
    const float e = __expf(s - m) * l;
    return j < nkey && s != -INFINITY ? e : 0.f;
  };
  {
    float mk[kPre], lk[kPre];
#pragma unroll
    for (int k = 0; k < kPre; ++k) {
      mk[k] = hm[min(hp + HP * k, nw - 1)];
      lk[k] = hl[min(hp + HP * k, nw - 1)];
    }
#pragma unroll
    for (int k = 0; k < kPre; ++k)
      if (hp + HP * k < nw) wt[(hp + HP * k) * CH + j] = weight(sv[k], mk[k], lk[k]);
  }
#pragma unroll 4
  for (int i = hp + HP * kPre; i < nw; i += HP) wt[i * CH + j] = weight(*score(i), hm[i], hl[i]);
  lds_sync();
  // ---- mixed weights of this kv head's columns (row, query head)
  {
    const int idx = ((j / M::KS) * 64 + 16 * ((j % M::KS) / M::EPL)) * M::EPL + j % M::EPL;
    // (the weights of eight heads are requested together, of one row for all of the wave's columns; a loop over the heads with the lane
    // read in it is not unrolled: an LDS round trip a head, 1.3 us of 16 heads in two columns -> 0.9)
    constexpr int GB = 8;
    float x[kCols] = {};
    if (in_lanes) {
#pragma unroll
      for (int i = 0; i < kCols; ++i) tk[i] = lane < p.H ? tk[i] : 0.f;
      for (int gb = 0; gb < p.H; gb += GB) {         // (heads past the last: a weight of 0)
        float wv[GB];
        auto read = [&](int row) {
#pragma unroll
          for (int u = 0; u < GB; ++u) wv[u] = wt[(row * hn + min(gb + u, p.H - 1)) * CH + j];
        };
        if constexpr (!GRP) read(0);
#pragma unroll
        for (int i = 0; i < kCols; ++i) {
          if (hp + HP * i >= ncol) break;              // (uniform per wave)
          if constexpr (GRP) read((hp + HP * i) / Rb);
#pragma unroll
          for (int u = 0; u < GB; ++u)
            x[i] += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, tk[i]), gb + u)) * wv[u];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
      const int cc = hp + HP * i, cr = GRP ? cc % Rb : cc;
      if (cc >= ncol) break;                         // (uniform per wave)
      const float* wr = wt + (GRP ? cc / Rb : 0) * hn * CH + j;
      if (!p.talk) {
        x[i] = wr[cr * CH];
      } else if (!in_lanes) {
        const float* t = p.talk + (size_t)(h0 + cr) * p.H;
#pragma unroll 8
        for (int g = 0; g < p.H; ++g) x[i] += t[g] * wr[g * CH];
      }
      stv(pf + idx + cc * M::EPL, x[i]);
    }
  }
  lds_sync();
  // ---- O^T = V^T . P^T
  const int nz = gridDim.z;
  float* prow = p.part + srow * p.nch * p.H * p.dv;
  const __amdgpu_buffer_rsrc_t rp = rsrc_f32(prow, (int64_t)p.nq * p.nch * p.H * p.dv);
  const float gate = on ? gate_of(p, ldv(&gate_raw)) : 0.f;
  for (int d = w * 16; d < p.dv; d += 16 * kWaves) {
    f32x4 acc = {};
#pragma unroll
    for (int s = 0; s < NST; ++s)
      if (s * TPS < nt) acc = M::mma(va[s], *reinterpret_cast<const uint4*>(pf + ((size_t)s * 64 + lane) * M::EPL), acc);
    if (d + 16 * kWaves < p.dv) load_v(d + 16 * kWaves);
    if (!col) continue;
    const int h = h0 + r;
    if (nact == 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) stv(out + (size_t)qi * p.ldo + (size_t)h * p.dv + d + 4 * b + i, on ? acc[i] * gate : 0.f);
    } else {
      st_sc1_x4(rp, (int)(((((int64_t)qi * p.nch + chunk) * p.H + h) * p.dv + d + 4 * b) * 4), acc);
    }
  }
  if (nact == 1) return;
  // ---- ticket; the last arriver adds the chunks in order
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    int* cnt = p.counters + ((size_t)ri * p.G + c) * nz + blockIdx.z;
    const int ticket = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = ticket == nact - 1;
    if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = last;
  }
  __syncthreads();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int per_row = Rb * p.dv;
  for (int i = threadIdx.x * 2; i < un.cnt * per_row; i += 2 * NT) {
    const int k0 = i / per_row, e = i % per_row, row = un.row + k0;
    const int64_t o = (int64_t)h0 * p.dv + e;
    float a0 = 0.f, a1 = 0.f;
#pragma unroll 8
    for (int k = 0; k < nact; ++k) {
      const float2 x = ld_sc1_f2(rp, ((int64_t)k0 * p.nch + k) * p.H * p.dv + o);
      a0 += x.x;
      a1 += x.y;
    }
    if (GRP && p.slots[row] < 0) {
      stv(out + (size_t)k0 * p.ldo + o, 0.f);
      stv(out + (size_t)k0 * p.ldo + o + 1, 0.f);
      continue;
    }
    const float g = gate_of(p, p.gate ? ldv(gate_at<T>(p, row, h0 + e / p.dv)) : 0.f);
    stv(out + (size_t)k0 * p.ldo + o, a0 * g);
    stv(out + (size_t)k0 * p.ldo + o + 1, a1 * g);
  }
}

// ------------------------------------------------------------------------------------------ prefill form
constexpr int kTab = 1024;                  // tiles a query tile may see (their cache places are kept in LDS)

// cache place of every visible tile: block * (tiles per block) + tile in the block
VWA_DEVICE void tile_table(const TalkAttnParams& p, const Vis& v, int seq, int* tab, int threads) {
  const int* gtab = p.block_table + (int64_t)seq * p.table_stride;
  const int lb = __builtin_ctz(p.block_size) - 4;           // log2 of the tiles per block
  for (int t = threadIdx.x; t < v.n; t += threads) {
    const int tl = tile_of(v, t);
    tab[t] = (gtab[tl >> lb] << lb) + (tl & ((1 << lb) - 1));
  }
}

// every key of the tile visible to every query p0 .. p1 (no per-key masks needed)
VWA_DEVICE bool all_visible(int p0, int p1, int key0, int window, int keep) {
  return key0 + kTile - 1 <= p0 && (window <= 0 || p1 - key0 < window || key0 + kTile - 1 < keep);
}

// Pass 1: log2-sum-exp of every (query, head): a workgroup per (16 queries, kv head, RB query heads),
// the query fragments in registers, its 4 waves taking every fourth key tile (next tile's keys in
// flight).  lse[row][H] = max + log2(sum) of the scaled scores in log2 units.
template <int RB, int KSN>
__global__ __launch_bounds__(256) void talk_lse_kernel(TalkPrefillParams pp) {
  const TalkAttnParams& p = pp.a;
  __shared__ float red[4][RB][16][2];
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, b = lane >> 4;
  const int lt = xcd_remap((int)blockIdx.x, pp.n_tiles * p.G);  // (a kv head's tiles share an XCD's L2)
  const int c = lt / pp.n_tiles, tile = lt % pp.n_tiles;
  const int row0 = pp.tiles[2 * tile], nq = pp.tiles[2 * tile + 1];
  const int R = p.H / p.G, r0 = blockIdx.y * RB, nr = min(RB, R - r0), nst = p.dk >> 5;
  const int pos0 = p.positions[row0], pos1 = pos0 + nq - 1, seq = p.seq_ids[row0];
  const int qrow = row0 + min(rl, nq - 1), qpos = pos0 + min(rl, nq - 1);
  const Vis v = vis_tiles(pos0, pos1, p.window, p.keep);
  const float sl2 = p.scale * kLog2e;
  __shared__ int tab[kTab];
  tile_table(p, v, seq, tab, 256);
  const int lb = __builtin_ctz(p.block_size) - 4;
  // (steps past dk: the query fragment is zero, the key fragment repeats the last step)
  uint4 qf[RB][KSN];
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int s = 0; s < KSN; ++s) {
      qf[r][s] = ld128(reinterpret_cast<const u16*>(p.q) + (size_t)qrow * p.ldq + (size_t)(c * R + r0 + min(r, nr - 1)) * p.dk +
                       b * 8 + min(s, nst - 1) * 32);
      if (s >= nst) qf[r][s] = make_uint4(0, 0, 0, 0);
    }
  __syncthreads();
  const u16* kbase = reinterpret_cast<const u16*>(p.k) + (int64_t)c * p.k_sh + rl * p.dk + b * 8;
  auto load_k = [&](uint4 (&kf)[KSN], int t) {
    const int ts = __builtin_amdgcn_readfirstlane(tab[min(t, v.n - 1)]);
    const u16* kp = kbase + (int64_t)(ts >> lb) * p.k_sb + (ts & ((1 << lb) - 1)) * kTile * p.dk;
#pragma unroll
    for (int s = 0; s < KSN; ++s) kf[s] = ld128(kp + min(s, nst - 1) * 32);
  };
  float m[RB], l[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    m[r] = -1e30f;
    l[r] = 0.f;
  }
  auto add_tile = [&](const uint4 (&kf)[KSN], int t) {
    const int key0 = tile_of(v, t) * kTile;
    const bool full = all_visible(pos0, pos1, key0, p.window, p.keep);
    bool vis[4] = {true, true, true, true};
    if (!full) {
#pragma unroll
      for (int i = 0; i < 4; ++i) vis[i] = sees(qpos, key0 + 4 * b + i, p.window, p.keep);
    }
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      f32x4 a = {};
#pragma unroll
      for (int s = 0; s < KSN; ++s) a = mfma16(as_bf16x8(kf[s]), as_bf16x8(qf[r][s]), a);
      float s[4], mn = m[r];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i] = vis[i] ? a[i] * sl2 : -1e30f;
        mn = fmaxf(mn, s[i]);
      }
      float x = l[r] * __builtin_amdgcn_exp2f(m[r] - mn);
#pragma unroll
      for (int i = 0; i < 4; ++i) x += vis[i] ? __builtin_amdgcn_exp2f(s[i] - mn) : 0.f;
      l[r] = x;
      m[r] = mn;
    }
  };
  uint4 ka[KSN], kb[KSN];
  load_k(ka, w);
  for (int t = w; t < v.n; t += 8) {
    load_k(kb, t + 4);
    add_tile(ka, t);
    if (t + 4 >= v.n) break;
    load_k(ka, t + 8);
    add_tile(kb, t + 4);
  }
#pragma unroll
  for (int r = 0; r < RB; ++r) {
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
      const float mo = __shfl_xor(m[r], o, 64), lo = __shfl_xor(l[r], o, 64), mn = fmaxf(m[r], mo);
      l[r] = l[r] * __builtin_amdgcn_exp2f(m[r] - mn) + lo * __builtin_amdgcn_exp2f(mo - mn);
      m[r] = mn;
    }
    if (b == 0) {
      red[w][r][rl][0] = m[r];
      red[w][r][rl][1] = l[r];
    }
  }
  __syncthreads();
  const int r = threadIdx.x >> 4, q = threadIdx.x & 15;
  if (r >= nr || q >= nq) return;
  float mm = -1e30f, ll = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) mm = fmaxf(mm, red[i][r][q][0]);
#pragma unroll
  for (int i = 0; i < 4; ++i) ll += red[i][r][q][1] * __builtin_amdgcn_exp2f(red[i][r][q][0] - mm);
  pp.lse[(size_t)(row0 + q) * p.H + c * R + r0 + r] = mm + __log2f(ll);
}

// Pass 2.  GP, RP: kv heads and query heads per kv head in the padded head order h = c * RP + r; NV: (kv
// head, 16 value columns) tiles per wave; KSN: 32-wide steps over the q / k dimensions.  8 waves walk
// the keys 32 (few heads: 64) at a time, in three stages with two barriers:
//   scores   a wave owns HW heads (their query fragments stay in its registers) and two key tiles; the
//            normalised weights x go to LDS as hi + lo bf16 pairs (16 mantissa bits together), in the
//            B-operand order of the mixing: k = (hi | lo, head), column = query, one block per key
//   mixing   a wave takes 4 keys: talk (bf16 as stored, repeated for both halves) times that block on
//            the MFMA; the mixed weights go back to LDS as bf16 in the B-operand order of the values
//   values   a wave owns NV value tiles of a kv head's query heads: O^T += V^T . P^T
// The values stage of one round and the scores of the next lie between the same two barriers.
// The tile's keys may be split over workgroups (blockIdx.y): their sums are added in order by the last
// one to finish.
constexpr int kPW = 8;                                               // waves
template <int GP, int RP, int NV, int KSN>
struct PrefillCfg {
  static constexpr int HT = GP * RP, HX = HT < 4 ? 4 : HT;
  static constexpr int KT = HX == 4 ? 4 : 2, KEYS = KT * kTile, KG = KT / 2;   // tiles, keys, 32-key groups per round
  static constexpr int HW = HX > kPW ? HX / kPW : 1;                 // heads per wave
  static constexpr int HWAVES = HX / HW;                             // waves over the heads; the others take other tiles
  static constexpr int NCW = HW > RP ? HW / RP : 1;                  // kv heads per wave
  static constexpr int MT = HT > 16 ? 2 : 1;                         // 16-row tiles of the mixed heads
  static constexpr int KM = HT > 16 ? 2 : 1;                         // 32-deep steps of the mixing
  // next keys requested after the values (not before the mixing): their registers would not fit beside
  // the accumulators and query fragments
  static constexpr bool LATE_K = NV * RP * 4 + HW * KSN * 4 > 128;
  static constexpr int NC = LATE_K ? (NV < 2 ? NV : 2) : NV < 4 ? NV : 4;   // value tiles loaded ahead
  static constexpr int X_BYTES = KEYS * KM * 1024, P_BYTES = HX * KEYS * 16 * 2;
  static constexpr int LDS = X_BYTES + P_BYTES + 2 * HX * 16 * 4 + kTab * 4;
};

// ONE: every wave's value tiles belong to one kv head (its mixed weights are read once per 32 keys)
template <int GP, int RP, int NV, int KSN, bool ONE>
__global__ __launch_bounds__(kPW * 64) void talk_prefill_kernel(TalkPrefillParams pp) {
  using C = PrefillCfg<GP, RP, NV, KSN>;
  constexpr int HT = C::HT, HX = C::HX, HW = C::HW, KG = C::KG, KT = C::KT;
  constexpr int HS = KG * 4 * 16 * 16;                               // bytes of a head's mixed weights
  constexpr int KB = C::KM * 1024;                                   // bytes of a key's mixing operand
  const TalkAttnParams& p = pp.a;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int s_last;
  char* xm = smem;                                                   // [KEYS][KM][64][16 B]
  char* pm = smem + C::X_BYTES;                                      // [HX][KG][4][16 q][8 keys]
  float* lse = reinterpret_cast<float*>(pm + C::P_BYTES);            // [HX][16]
  float* gate = lse + HX * 16;                                       // [HX][16] output factors
  int* btab = reinterpret_cast<int*>(gate + HX * 16);
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rl = lane & 15, b = lane >> 4;
  const int bt = xcd_remap((int)blockIdx.x, pp.n_tiles);
  const int row0 = pp.tiles[2 * bt], nq = pp.tiles[2 * bt + 1];
  const int R = p.H / p.G, nst = p.dk >> 5;
  const int pos0 = p.positions[row0], pos1 = pos0 + nq - 1, seq = p.seq_ids[row0];
  const int qrow = row0 + min(rl, nq - 1), qpos = pos0 + min(rl, nq - 1);
  const Vis v = vis_tiles(pos0, pos1, p.window, p.keep);
  const int nit = (v.n + KT - 1) / KT, per = (nit + pp.splits - 1) / pp.splits;
  const int nact = (nit + per - 1) / per;                            // splits with work
  const int split = blockIdx.y;
  if (split >= nact) return;
  const int it0 = split * per, it1 = min(nit, it0 + per);
  const float sl2 = p.scale * kLog2e;
  tile_table(p, v, seq, btab, kPW * 64);
  const int lb = __builtin_ctz(p.block_size) - 4, lm = (1 << lb) - 1;
  // (padding heads: weights exp2(-huge) = 0)
  for (int u = threadIdx.x; u < HX * 16; u += kPW * 64)
    if ((u >> 4) / RP >= p.G || (u >> 4) % RP >= R) lse[u] = 1e30f;
  for (int u = threadIdx.x; u < p.H * 16; u += kPW * 64) {
    const int h = u >> 4, q = u & 15;
    const int at = ((h / R) * RP + h % R) * 16 + q;
    lse[at] = pp.lse[(size_t)(row0 + min(q, nq - 1)) * p.H + h];
    gate[at] = gate_of(p, p.gate ? ldv(gate_at<u16>(p, row0 + min(q, nq - 1), h)) : 0.f);
  }
  // (operand slots no head writes -- padding heads, blocks past 2 HT -- stay zero)
  for (int u = threadIdx.x; u < C::X_BYTES / 16; u += kPW * 64) reinterpret_cast<uint4*>(xm)[u] = make_uint4(0, 0, 0, 0);
  // this wave's heads and tiles of a round
  const int hw0 = (w % C::HWAVES) * HW, tw0 = (w / C::HWAVES) * 2;
  const u16* qp = reinterpret_cast<const u16*>(p.q) + (size_t)qrow * p.ldq + b * 8;
  uint4 qf[HW][KSN];
  float ls[HW];
#pragma unroll
  for (int k = 0; k < HW; ++k) {
    const int c = min((hw0 + k) / RP, p.G - 1), r = min((hw0 + k) % RP, R - 1);
#pragma unroll
    for (int s = 0; s < KSN; ++s) {  // (steps past dk: zero here, the key fragment repeats the last step)
      qf[k][s] = ld128(qp + (size_t)(c * R + r) * p.dk + min(s, nst - 1) * 32);
      if (s >= nst) qf[k][s] = make_uint4(0, 0, 0, 0);
    }
  }
  uint4 tf[C::MT];                                                   // talk, A operand (both mixing steps use it)
#pragma unroll
  for (int mt = 0; mt < C::MT; ++mt) tf[mt] = reinterpret_cast<const uint4*>(pp.talk_frag)[mt * 64 + lane];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < HW; ++k) ls[k] = lse[(hw0 + k) * 16 + rl];
  const unsigned klane = rl * p.dk + b * 8;                          // (scalar tile base + one lane offset)
  auto load_k = [&](uint4 (&kf)[C::NCW][2][KSN], int it) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int ts = __builtin_amdgcn_readfirstlane(btab[min(it * KT + tw0 + u, v.n - 1)]);
      const u16* kp = reinterpret_cast<const u16*>(p.k) + (int64_t)(ts >> lb) * p.k_sb + (ts & lm) * kTile * p.dk;
#pragma unroll
      for (int c = 0; c < C::NCW; ++c)
#pragma unroll
        for (int s = 0; s < KSN; ++s)
          kf[c][u][s] = ld128(kp + (int64_t)min(hw0 / RP + c, p.G - 1) * p.k_sh + min(s, nst - 1) * 32 + klane);
    }
  };
  // value tiles of a wave in chunks of NC; a step is one chunk of one 32-key group
  const int ndv = p.dv >> 4, nvt = p.G * ndv, nvw = (nvt + kPW - 1) / kPW, v0 = w * nvw;
  constexpr int NC = C::NC, CH = NV / NC, STEPS = KG * CH;
  static_assert(NV % NC == 0, "whole chunks");
  // (value tiles past the last compute something nobody stores)
  auto tile_at = [&](int u) { return min(v0 + min(u, nvw - 1), nvt - 1); };
  const u16* vbase = reinterpret_cast<const u16*>(p.v) + rl * p.block_size + (b & 1) * 8;
  auto load_v = [&](uint4 (&vf)[NC], int it, int step) {
    const int ts = btab[min(it * KT + 2 * (step / CH) + (b >> 1), v.n - 1)];
    const u16* vp = vbase + (int64_t)(ts >> lb) * p.v_sb + (ts & lm) * kTile;
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      const int idx = tile_at((step % CH) * NC + n);
      vf[n] = ld128(vp + (int64_t)(idx / ndv) * p.v_sh + (int64_t)(idx % ndv) * 16 * p.block_size);
    }
  };

  f32x4 acc[NV][RP] = {};
  uint4 kf[C::NCW][2][KSN];
  load_k(kf, it0);
  // The values of a round's first step (two steps when there are several: va, vb) are requested at the end
  // of the round before it, its keys after the scores of the round before it
  static_assert(STEPS == 1 || STEPS % 2 == 0, "register sets by step parity");
  uint4 va[NC], vb[NC];
  load_v(va, it0, 0);
  if (STEPS > 1) load_v(vb, it0, 1);
  for (int it = it0; it < it1; ++it) {
    // ---- scores -> hi / lo weights
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = it * KT + tw0 + u;
      const int key0 = tile_of(v, min(t, v.n - 1)) * kTile;
      const bool ok = t < v.n, full = ok && all_visible(pos0, pos1, key0, p.window, p.keep);
      bool vis[4] = {true, true, true, true};
      if (!full) {
#pragma unroll
        for (int i = 0; i < 4; ++i) vis[i] = ok && sees(qpos, key0 + 4 * b + i, p.window, p.keep);
      }
      float x[HW][4];
#pragma unroll
      for (int k = 0; k < HW; ++k) {
        f32x4 a = {};
#pragma unroll
        for (int s = 0; s < KSN; ++s) a = mfma16(as_bf16x8(kf[k / RP][u][s]), as_bf16x8(qf[k][s]), a);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[k][i] = vis[i] ? __builtin_amdgcn_exp2f(a[i] * sl2 - ls[k]) : 0.f;
      }
      // head h, part (hi 0, lo 1) at byte: HT 32 part * 1024 + h / 8 block; 16 block 2 part + h / 8; 8 block
      // part; 4 block 0, element 4 part + h
      char* xw = xm + ((tw0 + u) * kTile + 4 * b) * KB + rl * 16 + (HX == 4 ? hw0 * 2 : (hw0 >> 3) * 256 + (hw0 & 7) * 2);
      constexpr int LO = HX == 32 ? 1024 : HX == 16 ? 512 : HX == 8 ? 256 : 8;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (HW == 1) {
          const u16 hi = f2bf(x[0][i]);
          *reinterpret_cast<u16*>(xw + i * KB) = hi;
          *reinterpret_cast<u16*>(xw + i * KB + LO) = f2bf(x[0][i] - bf2f(hi));
        } else {
          unsigned hi[HW / 2], lo[HW / 2];
#pragma unroll
          for (int k = 0; k < HW; k += 2) {
            hi[k / 2] = pack2(x[k][i], x[k + 1][i]);
            lo[k / 2] = pack2(x[k][i] - __uint_as_float(hi[k / 2] << 16), x[k + 1][i] - __uint_as_float(hi[k / 2] & 0xffff0000u));
          }
          if constexpr (HW == 2) {
            *reinterpret_cast<unsigned*>(xw + i * KB) = hi[0];
            *reinterpret_cast<unsigned*>(xw + i * KB + LO) = lo[0];
          } else {
            *reinterpret_cast<uint2*>(xw + i * KB) = make_uint2(hi[0], hi[1]);
            *reinterpret_cast<uint2*>(xw + i * KB + LO) = make_uint2(lo[0], lo[1]);
          }
        }
      }
    }
    lds_sync();
    if (!C::LATE_K) load_k(kf, it + 1);
    // ---- mixing: keys 4 kq .. 4 kq + 3
#pragma unroll
    for (int u = 0; u < KT / 2; ++u) {
      const int kq = w + 8 * u;
#pragma unroll
      for (int mt = 0; mt < C::MT; ++mt) {
        f32x4 y[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          y[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < C::KM; ++ks)
            y[g] = mfma16(as_bf16x8(tf[mt]), *reinterpret_cast<const bf16x8*>(xm + (4 * kq + g) * KB + ks * 1024 + lane * 16), y[g]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int h = 16 * mt + 4 * b + e;
          if (HX >= 16 || h < HX)
            *reinterpret_cast<uint2*>(pm + h * HS + (((kq >> 1) * 16) + rl) * 16 + (kq & 1) * 8) =
                make_uint2(pack2(y[0][e], y[1][e]), pack2(y[2][e], y[3][e]));
        }
      }
    }
    lds_sync();
    // ---- values
    auto load_p = [&](uint4 (&pf)[RP], int c, int kg) {
#pragma unroll
      for (int r = 0; r < RP; ++r)
        pf[r] = *reinterpret_cast<const uint4*>(pm + (c * RP + r) * HS + ((kg * 4 + b) * 16 + rl) * 16);
    };
    uint4 pf[RP];
#pragma unroll
    for (int st = 0; st < STEPS; ++st) {
      const int kg = st / CH;
      if (kg > 0 && it * KT + 2 * kg >= v.n) break;
      uint4(&vc)[NC] = st & 1 ? vb : va;
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        const int u = (st % CH) * NC + n;
        // (a kv head's mixed weights serve all of this wave's value tiles of it)
        if (u == 0 || (!ONE && tile_at(u) / ndv != tile_at(u - 1) / ndv)) load_p(pf, tile_at(u) / ndv, kg);
#pragma unroll
        for (int r = 0; r < RP; ++r) acc[u][r] = mfma16(as_bf16x8(vc[n]), as_bf16x8(pf[r]), acc[u][r]);
      }
      // the step after next (or the next round's) into the registers just used
      if (STEPS == 1) load_v(vc, it + 1, 0);
      else load_v(vc, st + 2 < STEPS ? it : it + 1, st + 2 < STEPS ? st + 2 : st + 2 - STEPS);
    }
    if (C::LATE_K) load_k(kf, it + 1);
  }
  if (nact > 1) {
    // ---- every split's sums out (sc1), a ticket, and the last one adds them in order
    constexpr int kWave = NV * RP * 64 * 16, kPart = kPW * kWave;     // bytes per wave / workgroup
    float* base = pp.part + (size_t)bt * pp.splits * (kPart / 4);
    const __amdgpu_buffer_rsrc_t rp = rsrc_f32(base, (int64_t)pp.splits * (kPart / 4));
    const int at = w * kWave + lane * 16;
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int r = 0; r < RP; ++r) st_sc1_x4(rp, split * kPart + at + (n * RP + r) * 1024, acc[n][r]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
      const int ticket = __hip_atomic_fetch_add(pp.tickets + bt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = ticket == nact - 1;
      if (last) __hip_atomic_store(pp.tickets + bt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = last;
    }
    __syncthreads();
    if (!s_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int r = 0; r < RP; ++r) acc[n][r] = ld_sc1_x4(rp, at + (n * RP + r) * 1024);
    for (int s = 1; s < nact; ++s)
#pragma unroll
      for (int n = 0; n < NV; ++n)
#pragma unroll
        for (int r = 0; r < RP; ++r) acc[n][r] += ld_sc1_x4(rp, s * kPart + at + (n * RP + r) * 1024);
  }
  // ---- gate, scale, store: lane (query rl, value columns 4b .. 4b+3 of the tile)
  if (rl >= nq) return;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const int idx = v0 + n;
    if (n >= nvw || idx >= nvt) break;
    const int c = idx / ndv, d = (idx % ndv) * 16 + 4 * b;
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      if (r >= R) break;
      const int h = c * R + r;
      const float g = gate[(c * RP + r) * 16 + rl];
      uint2 o;
      o.x = pack2(acc[n][r][0] * g, acc[n][r][1] * g);
      o.y = pack2(acc[n][r][2] * g, acc[n][r][3] * g);
      *reinterpret_cast<uint2*>(reinterpret_cast<u16*>(p.out) + (size_t)qrow * p.ldo + (size_t)h * p.dv + d) = o;
    }
  }
}

int pow2_up(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

constexpr size_t kMaxLds = 160 * 1024;

// what a call wants: only whether the sizes have an instantiation, its partial floats per tile and split,
// or the launch
enum Want { WANT_FIT, WANT_PART, WANT_LAUNCH };

template <int GP, int RP, int NV, int KSN>
int64_t prefill_cfg(const TalkPrefillParams& p, hipStream_t st, Want want) {
  using C = PrefillCfg<GP, RP, NV, KSN>;
  static_assert(C::LDS <= kMaxLds - 64, "LDS");
  if (want == WANT_FIT) return 0;
  if (want == WANT_PART) return (int64_t)kPW * NV * RP * 256;
  const int R = p.a.H / p.a.G;
  constexpr int RB = RP < 4 ? RP : 4;
  hipLaunchKernelGGL((talk_lse_kernel<RB, KSN>), dim3(p.n_tiles * p.a.G, (R + RB - 1) / RB), dim3(256), 0, st, p);
  const dim3 grid(p.n_tiles, p.splits), block(kPW * 64);
  if constexpr (KSN == 4 && NV == GP) {  // (the usual sizes)
    const int ndv = p.a.dv >> 4, nvw = (p.a.G * ndv + kPW - 1) / kPW;
    if (ndv % nvw == 0) {
      hipLaunchKernelGGL((talk_prefill_kernel<GP, RP, NV, KSN, true>), grid, block, C::LDS, st, p);
      return 0;
    }
  }
  hipLaunchKernelGGL((talk_prefill_kernel<GP, RP, NV, KSN, false>), grid, block, C::LDS, st, p);
  return 0;
}

template <int GP, int RP>
int64_t prefill_sizes(const TalkPrefillParams& p, hipStream_t st, Want want) {
  constexpr int N1 = GP, N2 = 2 * GP;   // value tiles per wave: dv <= 128 / <= 256
  const int need = (p.a.G * (p.a.dv >> 4) + kPW - 1) / kPW;
  if (need <= N1) {
    if (p.a.dk <= 64) return prefill_cfg<GP, RP, N1, 2>(p, st, want);
    if (p.a.dk <= 128) return prefill_cfg<GP, RP, N1, 4>(p, st, want);
    return prefill_cfg<GP, RP, N1, 8>(p, st, want);
  }
  if constexpr (GP * RP <= 16) {
    if (need <= N2) {
      if (p.a.dk <= 64) return prefill_cfg<GP, RP, N2, 2>(p, st, want);
      if (p.a.dk <= 128) return prefill_cfg<GP, RP, N2, 4>(p, st, want);
      return prefill_cfg<GP, RP, N2, 8>(p, st, want);
    }
  }
  return -10;
}

int64_t dispatch_prefill(const TalkPrefillParams& p, hipStream_t st, Want want) {
  const TalkAttnParams& a = p.a;
  if (a.H < 1 || a.G < 1 || a.H % a.G || a.dk % 32 || a.dk > 256 || a.dv % 16 || a.dv < 16) return -10;
  switch (pow2_up(a.G) * 100 + pow2_up(a.H / a.G)) {
    case 101: return prefill_sizes<1, 1>(p, st, want);
    case 102: return prefill_sizes<1, 2>(p, st, want);
    case 104: return prefill_sizes<1, 4>(p, st, want);
    case 108: return prefill_sizes<1, 8>(p, st, want);
    case 201: return prefill_sizes<2, 1>(p, st, want);
    case 202: return prefill_sizes<2, 2>(p, st, want);
    case 204: return prefill_sizes<2, 4>(p, st, want);
    case 208: return prefill_sizes<2, 8>(p, st, want);
    case 401: return prefill_sizes<4, 1>(p, st, want);
    case 402: return prefill_sizes<4, 2>(p, st, want);
    case 404: return prefill_sizes<4, 4>(p, st, want);
    case 408: return prefill_sizes<4, 8>(p, st, want);
    case 801: return prefill_sizes<8, 1>(p, st, want);
    case 802: return prefill_sizes<8, 2>(p, st, want);
    case 804: return prefill_sizes<8, 4>(p, st, want);
    case 1601: return prefill_sizes<16, 1>(p, st, want);
    case 1602: return prefill_sizes<16, 2>(p, st, want);
    default: return -10;
  }
}

int check_attn(const TalkAttnParams& p) {
  if (p.rows < 1 || p.G < 1 || p.H < 1 || p.H % p.G || p.block_size < kTile || (p.block_size & (p.block_size - 1)) || p.dk % 32 || p.dv % 16) return -1;
  if (p.window < 0 || p.keep < 0) return -2;
  if ((p.k_sh | p.k_sb | p.v_sh | p.v_sb | p.ldq) % 8) return -3;
  return 0;
}

template <class T, int CT, bool GRP>
int launch_rows(const TalkAttnParams& p, hipStream_t st, const QkvCacheParams* qc = nullptr, const MinGruParams* g = nullptr) {
  const size_t lds = mix_lds<T, CT>(p.H, p.nq);
  if (lds > kMaxLds - 64) return -5;
  const int nz = (p.H / p.G + 15) / 16;
  if (qc) {
    const int n = p.rows * p.G * nz, per_row = step_wgs(n, p.nst);
    hipLaunchKernelGGL((talk_step_kernel<T>), dim3(p.rows * (kStepParts + (g->width + 255) / 256) + n * per_row), dim3(256), 0, st, p, *qc, *g, per_row);
  } else
    hipLaunchKernelGGL((talk_scores_kernel<T, GRP>), dim3(p.rows * p.G, p.nst, nz), dim3(256), 0, st, p);
  hipLaunchKernelGGL((talk_mix_kernel<T, CT, GRP>), dim3(p.rows * p.G, p.nch, nz), dim3(64 * kWaves), lds, st, p);
  return (int)hipGetLastError();
}

}  // namespace

extern "C" int vwa_talk_attention(const TalkAttnParams* p, hipStream_t st) {
  const int rc = check_attn(*p);
  if (rc) return rc;
  if (p->nch < 1 || p->nst < 1 || !p->s || !p->stat || !p->part || !p->counters) return -4;
  if (p->nq < 1 || (int64_t)p->nq * p->nch * p->H * p->dv * 4 >= (1ll << 31)) return -5;
  if (p->groups) {
    if (p->nq * (p->H / p->G) > 16) return -6;
    return p->f32 ? launch_rows<float, 8, true>(*p, st) : launch_rows<u16, 8, true>(*p, st);
  }
  if (p->nq != 1) return -6;
  if (talk_chunk_tiles(p->H, 0) == 16) return p->f32 ? launch_rows<float, 16, false>(*p, st) : launch_rows<u16, 16, false>(*p, st);
  return p->f32 ? launch_rows<float, 8, false>(*p, st) : launch_rows<u16, 8, false>(*p, st);
}

// Scoring workgroups of a row, kv head and 16 query heads in vwa_talk_step, of n such and so many chunks of tiles
extern "C" int vwa_talk_step_wgs(int n, int chunks) { return n < 1 || chunks < 1 ? 0 : step_wgs(n, chunks); }

extern "C" int vwa_talk_step(const TalkAttnParams* p, const QkvCacheParams* qc, const MinGruParams* g, hipStream_t st) {
  const int rc = check_attn(*p);
  if (rc) return rc;
  if (p->nch < 1 || p->nst < 1 || !p->s || !p->stat || !p->part || !p->counters) return -4;
  if (p->nq != 1 || p->groups || p->row_list || (int64_t)p->nch * p->H * p->dv * 4 >= (1ll << 31)) return -5;
  if (p->rows > 64 || qc->rows != p->rows || g->rows != p->rows || g->width < 1 || qc->f32 != p->f32 || g->f32 != p->f32) return -6;
  if (qc->H != p->H || qc->G != p->G || qc->dk != p->dk || qc->dv != p->dv || qc->k != p->k || qc->v != p->v ||
      qc->block_size != p->block_size) return -7;
  if (qc->rot_dims < 16 || qc->rot_dims > qc->dk || qc->rot_dims % 16 || qc->max_pos < 1 || qc->ldx % 8 ||
      ((reinterpret_cast<uintptr_t>(qc->rope) | reinterpret_cast<uintptr_t>(qc->x)) & 15)) return -8;
  if (talk_chunk_tiles(p->H, 0) == 16) return p->f32 ? launch_rows<float, 16, false>(*p, st, qc, g) : launch_rows<u16, 16, false>(*p, st, qc, g);
  return p->f32 ? launch_rows<float, 8, false>(*p, st, qc, g) : launch_rows<u16, 8, false>(*p, st, qc, g);
}

extern "C" int64_t vwa_talk_prefill_part(int H, int G, int dk, int dv) {
  TalkPrefillParams p{};
  p.a.H = H;
  p.a.G = G;
  p.a.dk = dk;
  p.a.dv = dv;
  return dispatch_prefill(p, nullptr, WANT_PART);
}

extern "C" int vwa_talk_prefill(const TalkPrefillParams* p, hipStream_t st) {
  const int rc = check_attn(p->a);
  if (rc) return rc;
  if (p->max_tiles < 1 || p->max_tiles > kTab) return -8;  // (the kernel keeps the tiles' places in LDS)
  if (p->a.f32 || p->n_tiles < 1 || !p->tiles || !p->talk_frag || !p->lse || p->splits < 1 || p->a.ldo % 4) return -6;
  if (p->splits > 1) {
    const int64_t part = dispatch_prefill(*p, st, WANT_PART);
    if (!p->part || !p->tickets || part < 0 || part * p->splits * 4 >= (1ll << 31)) return -7;
  }
  const int64_t r = dispatch_prefill(*p, st, WANT_LAUNCH);
  if (r) return (int)r;
  return (int)hipGetLastError();
}
