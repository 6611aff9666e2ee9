// Pieces shared by the persistent Whisper decoder kernels (whisper_dec.hip, whisper_dec_narrow.hip): LDS
// layout, loads and stores that cross workgroups inside a launch, level counters, the cross K / V prefetch, block reductions.
#pragma once
#include "common.h"
#include "vwa_kernels.h"

namespace {
using namespace vwa;

constexpr int kT = 512;           // threads (8 waves, K split over the waves)
constexpr int kSlots = 5, kLps = 5;
enum { LV_QKV = 0, LV_XQX, LV_SATT, LV_OXQ, LV_XATT, LV_XO, LV_FC1, LV_FC2 };
// gemm ids (WdecLayer::g; a slot's kind): the level of each
enum { G_QKV = 0, G_O, G_XQ, G_XO, G_FC1, G_FC2, G_XQO };
// role row layout (kWdRole ints per workgroup)
enum { R_KIND = 0, R_TILE = 5, R_PART = 10, R_RELOAD = 15, R_SATT = 20, R_XATT = 21, R_XPRE = 22, R_WORK = 23 };
// LDS layout (bytes)
constexpr int L_XS = 0;          // bf16 activation row (<= 5120)
constexpr int L_RED = 10368;     // f32 [8][32] cross-wave partial sums of a level's <= 2 tiles
constexpr int L_STAT = 11392;    // f32 [16]: mean, rstd
constexpr int L_W8 = 11456;      // f32 [2][8] per-wave reduction values
constexpr int L_QF = 11520;      // f32 [64] query head
constexpr int L_P = 11776;       // f32 [512] attention weights
constexpr int L_OW = 13824;      // f32 [8][64] per-wave attention outputs
constexpr int L_VA = 15872;      // int [512] self-attention K / V row offsets (elements)
constexpr int L_KV = 65536;      // cross-attention K chunk [<= 384][64] bf16, V chunk at + 48 KB
constexpr int L_KVV = 49152;
constexpr int kLds = 163840;
constexpr int kMaxChunk = 384;
constexpr int kSpinLimit = 1 << 17;  // bounded polls: a non-resident producer ends the launch, not the GPU
constexpr int kErrWord = 1024;       // (WdecParams::cnt u64 index of the error flag)
constexpr int kHeadCnt = 1280;      // (u64 index: per-head QKV completion counters, 128 B apart, <= 48 heads)
constexpr int kSmpCnt = 1152;       // (u64 index: the fused sampler's arrival counters, 8 groups x 128 B, monotonic)

// Wave-uniform values through readfirstlane.  The per-layer descriptors are read with VECTOR loads
// (the kernel stores to global memory, so the compiler cannot prove them unclobbered for scalar
// loads): a buffer resource built from such a pointer lives in VGPRs, and every buffer load through
// it became a waterfall loop -- readfirstlane / compare / exec loop with a vmcnt(0) per iteration,
// i.e. each 1 KB weight load of a refill and each self-attention V load waited for every load
// before it (60 such loads in the ISA).  Every pointer and size here is uniform by construction.
VWA_DEVICE int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T>
VWA_DEVICE T* uni(T* p) {
  const unsigned long long v = reinterpret_cast<unsigned long long>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
  return reinterpret_cast<T*>(((unsigned long long)hi << 32) | lo);
}

VWA_DEVICE __amdgpu_buffer_rsrc_t rsrc_of(const void* p, long long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(uni(const_cast<void*>(p)), (short)0,
                                           uni((int)(bytes < 0x7FFFFFF0ll ? bytes : 0x7FFFFFF0ll)), 0x00020000);
}

// sc1 (device-coherent) loads / stores of data crossing workgroups inside the launch
VWA_DEVICE uint4 ld_sc1_b128(__amdgpu_buffer_rsrc_t r, unsigned off) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 16);
  return make_uint4(v.x, v.y, v.z, v.w);
}
VWA_DEVICE void st_sc1_b128(__amdgpu_buffer_rsrc_t r, unsigned off, const uint4& v) {
  __builtin_amdgcn_raw_buffer_store_b128(u32x4{v.x, v.y, v.z, v.w}, r, (int)off, 0, 16);
}
VWA_DEVICE float ldf_sc1(const float* p) { return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
VWA_DEVICE void stf_sc1(float* p, float v) { __hip_atomic_store(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
VWA_DEVICE u16 ldh_sc1(const u16* p) { return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
VWA_DEVICE void sth_sc1(u16* p, u16 v) { __hip_atomic_store(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

VWA_DEVICE void set_err(const WdecParams& p) {
  __hip_atomic_store(gp(p.cnt + kErrWord), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sum of a level's eight group counters in one scalar round trip (glc: past the scalar cache)
VWA_DEVICE unsigned long long cnt_sum8(const unsigned long long* c) {
  unsigned long long v0, v1, v2, v3, v4, v5, v6, v7;
  asm volatile(
      "s_load_dwordx2 %0, %8, 0x0 glc\n\t"
      "s_load_dwordx2 %1, %8, 0x80 glc\n\t"
      "s_load_dwordx2 %2, %8, 0x100 glc\n\t"
      "s_load_dwordx2 %3, %8, 0x180 glc\n\t"
      "s_load_dwordx2 %4, %8, 0x200 glc\n\t"
      "s_load_dwordx2 %5, %8, 0x280 glc\n\t"
      "s_load_dwordx2 %6, %8, 0x300 glc\n\t"
      "s_load_dwordx2 %7, %8, 0x380 glc\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&s"(v0), "=&s"(v1), "=&s"(v2), "=&s"(v3), "=&s"(v4), "=&s"(v5), "=&s"(v6), "=&s"(v7)
      : "s"(c)
      : "memory");
  return v0 + v1 + v2 + v3 + v4 + v5 + v6 + v7;
}

VWA_DEVICE unsigned long long* lvl_cnt(const WdecParams& p, int lvl) { return p.cnt + (size_t)lvl * 8 * 16; }

// wave 0 polls until the level's counters reach target; bounded (a timed-out spin sets the error
// word: that step's results are invalid, the host falls back to per-kernel launches)
VWA_DEVICE void wd_wait(const WdecParams& p, int lvl, unsigned long long target) {
  if (VWA_TX < 64) {
    const unsigned long long* c = lvl_cnt(p, lvl);
    int spins = 0;
    while ((long long)(cnt_sum8(c) - target) < 0) {
      __builtin_amdgcn_s_sleep(1);
      // another workgroup already gave up: this launch is invalid anyway -- do not spin out again
      if ((spins & 255) == 255 && __hip_atomic_load(gp(p.cnt + kErrWord), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        break;
      if (++spins > kSpinLimit) {
        if (VWA_TX == 0) set_err(p);
        break;
      }
    }
  }
  lds_sync();
}

// this workgroup completed level lvl: every wave's stores are performed, then one no-return add on
// the group counter
VWA_DEVICE void wd_arrive(const WdecParams& p, int lvl) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  lds_sync();
  if (VWA_TX == 0)
    __hip_atomic_fetch_add(gp(lvl_cnt(p, lvl) + 16 * (blockIdx.x & 7)), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// diagnostic stamp k of (layer, level) (tools/wdec_probe.py): 0 entry, 1 released, 2 row staged
// (attention levels of whisper_dec.hip: softmax done), 3 completed
VWA_DEVICE void wd_stamp(const WdecParams& p, int li, int lvl, int k) {
  if (p.ts && VWA_TX == 0)
    *gp(p.ts + ((size_t)blockIdx.x * p.n_layers * kWdLevels + (size_t)li * kWdLevels + lvl) * 4 + k) =
        __builtin_amdgcn_s_memrealtime();
}

// cross-attention K / V chunk of layer li (this workgroup's item) -> LDS by LDS-DMA (no registers;
// completes on vmcnt: the level waits for it)
VWA_DEVICE void wd_kv_prefetch(const WdecParams& p, int li, int item, char* lds) {
  const int h = item / p.nch, ch = item % p.nch;
  const int k0 = ch * p.ch_len, nk = min(p.ch_len, p.T - k0);
  const int sess = p.cross_table[p.seq_ids[0]];
  const WdecLayer& L = p.layers[li];
  const long long bytes = (long long)p.sessions * p.T * p.H * 64 * 2;
  const __amdgpu_buffer_rsrc_t rk = rsrc_of(L.xk, bytes), rv = rsrc_of(L.xv, bytes);
  const int tx = VWA_TX, lane = tx & 63, w = uni(tx >> 6);  // (uniform: the K / V select stays scalar)
  const int n8 = (nk + 7) >> 3;  // 1 KB instructions (8 keys of 128 B) per tensor
  for (int r = w; r < 2 * n8; r += 8) {
    const bool isv = r >= n8;
    const int rr = isv ? r - n8 : r;
    const int kk = rr * 8 + (lane >> 3);
    // K rows XOR-swizzled by 16-byte chunk (LDS slot j of key kk holds chunk j ^ (kk & 7)): the
    // key-per-thread dot products read 8 different bank groups per 8 lanes instead of one
    const int chunk = isv ? (lane & 7) : ((lane & 7) ^ (kk & 7));
    const unsigned off = kk < nk ? (unsigned)(((((long long)sess * p.T + k0 + kk) * p.H + h) * 64 + chunk * 8) * 2)
                                 : 0x7FFFFFF0u;
    auto* dst = (__attribute__((address_space(3))) void*)(lds + L_KV + (isv ? L_KVV : 0) + rr * 1024);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(isv ? rv : rk, dst, 16, off, 0, 0, 0);
  }
}

// block-wide max / sum of one value per thread (all threads get the result)
VWA_DEVICE float blk_max(char* lds, float v) {
  float* w8 = reinterpret_cast<float*>(lds + L_W8);
  v = wave_max(v);
  if ((VWA_TX & 63) == 0) w8[VWA_TX >> 6] = v;
  lds_sync();
  float m = w8[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) m = fmaxf(m, w8[i]);
  return m;
}
VWA_DEVICE float blk_sum(char* lds, float v) {
  float* w8 = reinterpret_cast<float*>(lds + L_W8) + 8;
  v = wave_sum(v);
  if ((VWA_TX & 63) == 0) w8[VWA_TX >> 6] = v;
  lds_sync();
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) s += w8[i];
  return s;
}

// softmax over the thread-per-key scores s (keys t < nk, others -inf): returns (max, sum); P[t] in LDS
// (w8 max slots [0, 8) and sum slots [8, 16) are distinct: no barrier between the two reductions)
VWA_DEVICE float2 wd_softmax(char* lds, float s, bool valid) {
  float* P = reinterpret_cast<float*>(lds + L_P);
  const float m = blk_max(lds, valid ? s : -INFINITY);
  const float e = valid ? __expf(s - m) : 0.f;
  P[VWA_TX] = e;
  const float l = blk_sum(lds, e);  // (its barrier publishes P)
  return make_float2(m, l);
}

// per-wave partial outputs (lane = dim) -> LDS, summed by threads < 64 after the barrier
VWA_DEVICE float wd_ow_sum(char* lds, float o) {
  float* ow = reinterpret_cast<float*>(lds + L_OW);
  const int tx = VWA_TX;
  ow[(tx >> 6) * 64 + (tx & 63)] = o;
  lds_sync();
  float s = 0.f;
  if (tx < 64) {
#pragma unroll
    for (int w = 0; w < 8; ++w) s += ow[w * 64 + tx];
  }
  return s;
}

VWA_DEVICE void argmax_merge(float& bv, int& bi, float v, int i) {
  if (v > bv || (v == bv && i < bi)) {  // (sample.hip's order: the lowest id on ties)
    bv = v;
    bi = i;
  }
}

// the sampled token into the device loop's state (decode_advance_kernel's arithmetic)
VWA_DEVICE void wd_advance(const WdecParams& p, int tok) {
  p.smp_tok[0] = tok;
  p.smp_step[0] += 1;
  const int c = p.loop_cnt[0];
  if (c < p.loop_max) p.loop_out[c] = tok;
  p.loop_cnt[0] = c + 1;
  p.adv_tokens[0] = tok;
  const int pos = p.adv_positions[0] + 1;
  p.adv_positions[0] = pos;
  p.adv_ctx[0] = pos + 1;
  p.adv_slots[0] = (int64_t)(p.loop_base_block + pos / p.block_size) * p.block_size + pos % p.block_size;
}

}  // namespace
