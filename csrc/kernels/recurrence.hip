// Gated recurrences (f32 state per sequence and channel, one state slot per live sequence).
//
// minGRU: z = sigmoid(zp + zb), u = xp + xb, S <- (1 - z) S + z * (u >= 0 ? u + 1/2 : sigmoid(u)),
// out = S * silu(gp) * out_scale.  The gates read only the current token, so a run of tokens is a
// first-order linear scan per channel:
//
//  * rows form (decode steps, <= 64 rows): one workgroup per (256 channels, run of rows of one
//    sequence); the run's head row walks it token by token;
//  * scan form (prompt-sized runs): runs are cut into chunks.  Launch 1 reduces each chunk to
//    S_end = A S_start + B (and takes a copy of the run's initial state); launch 2 folds the chunks
//    in front of its own, then walks its tokens and writes the outputs; the run's last chunk
//    writes the state back.  Two streaming passes over the projections, all chunks in parallel.
//
// A run that starts at position 0 starts from a zero state whatever the slot holds.
#include "recurrence.h"

using namespace vwa;

namespace {

template <class T>
__global__ __launch_bounds__(256) void mingru_rows_kernel(MinGruParams p) {
  mingru_row<T>(p, blockIdx.y, blockIdx.x * 256 + threadIdx.x);
}

constexpr int kScanBatch = 8;  // rows whose loads are in flight together, a batch ahead of the arithmetic

constexpr int kFold = 16;      // chunks in front that are folded together

// PASS 1: per (chunk, channel) A = prod (1 - z), B = the chunk's end state from a zero start
// PASS 2: outputs (and the state of a run's last chunk)
// PAIRS (even widths whose columns pair up to a load): z c is added unrounded, else (1 - z) S (min_gru_step); the two were different kernels
// once, and their results stay what they were.
// A thread a channel.  Bound by a chunk's chain of rows and, with many chunks, by the exact exponentials and divisions of the gates: what
// counts is threads.  us of both passes, two channels a thread (and the chunks in front by sixteens, the rest of them one by one) ->
// here: 777 rows x 1024 in 32 bits 33.3 -> 16.5, 200 x 2048 in 16 bits 26.9 -> 17.4, 2048 x 4096 57 -> 42.5, 7200 x 1024 (pass 2) 24.8 -> 16.8.
template <class T, int PASS, bool PAIRS>
__global__ __launch_bounds__(256) void mingru_scan_kernel(MinGruParams p) {
  const int ck = blockIdx.y, ch = blockIdx.x * 256 + threadIdx.x;
  if (ch >= p.width) return;
  const int row0 = p.chunks[4 * ck], n = p.chunks[4 * ck + 1], idx = p.chunks[4 * ck + 2], cnt = p.chunks[4 * ck + 3];
  const T* z = reinterpret_cast<const T*>(p.z) + ch + (size_t)row0 * p.ld;
  const T* x = reinterpret_cast<const T*>(p.x) + ch + (size_t)row0 * p.ld;
  const T* g = reinterpret_cast<const T*>(p.g) + ch + (size_t)row0 * p.ld;
  const float zb = p.zb ? p.zb[ch] : 0.f, xb = p.xb ? p.xb[ch] : 0.f;
  float S = 0.f, A = 1.f;
  float bz[2][kScanBatch], bx[2][kScanBatch], bg[2][kScanBatch];
  auto load = [&](int q, int t0) {
#pragma unroll
    for (int t = 0; t < kScanBatch; ++t) {
      const size_t o = (size_t)min(t0 + t, n - 1) * p.ld;
      bz[q][t] = ldv(z + o);
      bx[q][t] = ldv(x + o);
      if (PASS == 2) bg[q][t] = ldv(g + o);
    }
  };
  load(0, 0);
  float* st = p.state + (size_t)p.seq_ids[row0] * p.state_ld + ch;
  const size_t W = p.width;
  if constexpr (PASS == 2) {
    // the chunks in front, a batch's loads in flight together (places past the last are read again)
    const int first = ck - idx;
    S = p.cS[first * W + ch];
    for (int k = first; k < ck; k += kFold) {
      float a[kFold], b[kFold];
#pragma unroll
      for (int f = 0; f < kFold; ++f) {
        const size_t o = min(k + f, ck - 1) * W + ch;
        a[f] = p.cA[o];
        b[f] = p.cB[o];
      }
#pragma unroll
      for (int f = 0; f < kFold; ++f) S = k + f < ck ? a[f] * S + b[f] : S;
    }
  }
  T* out = reinterpret_cast<T*>(p.out) + (size_t)row0 * p.ldo + ch;
  auto work = [&](int q, int t0) {
#pragma unroll
    for (int t = 0; t < kScanBatch; ++t) {
      if (t0 + t >= n) break;
      const Gate gt = min_gru_gate(bz[q][t] + zb, bx[q][t] + xb);
      A *= 1.f - gt.z;
      S = PAIRS ? fmaf(gt.z, gt.c, (1.f - gt.z) * S) : min_gru_step(gt, S);
      if (PASS == 2) stv(out + (size_t)(t0 + t) * p.ldo, S * silu(bg[q][t]) * p.out_scale);
    }
  };
  for (int t0 = 0; t0 < n; t0 += 2 * kScanBatch) {
    if (t0 + kScanBatch < n) load(1, t0 + kScanBatch);
    work(0, t0);
    if (t0 + kScanBatch >= n) break;
    if (t0 + 2 * kScanBatch < n) load(0, t0 + 2 * kScanBatch);
    work(1, t0 + kScanBatch);
  }
  if constexpr (PASS == 1) {
    p.cA[ck * W + ch] = A;
    p.cB[ck * W + ch] = S;
    if (idx == 0) p.cS[ck * W + ch] = p.positions[row0] > 0 ? *st : 0.f;
  } else {
    if (idx == cnt - 1) *st = S;
  }
}

template <class T, bool PAIRS>
void launch_scan(const MinGruParams& p, hipStream_t st) {
  const dim3 grid((p.width + 255) / 256, p.n_chunks), block(256);
  hipLaunchKernelGGL((mingru_scan_kernel<T, 1, PAIRS>), grid, block, 0, st, p);
  hipLaunchKernelGGL((mingru_scan_kernel<T, 2, PAIRS>), grid, block, 0, st, p);
}

}  // namespace

extern "C" int vwa_mingru_rows(const MinGruParams* p, hipStream_t st) {
  if (p->rows < 1 || p->width < 1) return -1;
  const dim3 grid((p->width + 255) / 256, p->rows), block(256);
  if (p->f32) hipLaunchKernelGGL((mingru_rows_kernel<float>), grid, block, 0, st, *p);
  else hipLaunchKernelGGL((mingru_rows_kernel<u16>), grid, block, 0, st, *p);
  return (int)hipGetLastError();
}

extern "C" int vwa_mingru_scan(const MinGruParams* p, hipStream_t st) {
  if (p->rows < 1 || p->width < 1 || p->n_chunks < 1 || !p->chunks || !p->cA || !p->cB || !p->cS) return -1;
  const uintptr_t al = p->f32 ? 7 : 3;
  const bool pairs = p->width % 2 == 0 && p->ld % 2 == 0 && !((reinterpret_cast<uintptr_t>(p->z) | reinterpret_cast<uintptr_t>(p->x) |
                                                               reinterpret_cast<uintptr_t>(p->g)) & al);
  if (p->f32) pairs ? launch_scan<float, true>(*p, st) : launch_scan<float, false>(*p, st);
  else pairs ? launch_scan<u16, true>(*p, st) : launch_scan<u16, false>(*p, st);
  return (int)hipGetLastError();
}
