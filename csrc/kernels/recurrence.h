// Device parts of the gated recurrences, shared by their own launches (recurrence.hip) and the fused
// decode launch (stack_ops.hip).
#pragma once
#include "common.h"
#include "stack_kernels.h"
#include "stack_types.h"

namespace {
using namespace vwa;

struct Gate {
  float z, c;
};
VWA_DEVICE Gate min_gru_gate(float zp, float u) {
  return Gate{sigm(zp), u >= 0.f ? u + 0.5f : sigm(u)};
}
// (1 - z) S + z c with one product rounded before the sum.  Written out: which one it is was the compiler's choice, and code around it
// changed the choice and with it the bits of whole answers.
VWA_DEVICE float min_gru_step(const Gate& g, float S) { return fmaf(1.f - g.z, S, g.z * g.c); }

// Rows form of one (row, channel): the head row of a run of its sequence walks the run.  A decoded row is three round trips long:
// the ids of the row and its neighbours with its projections, the state, the results.
template <class T>
VWA_DEVICE void mingru_row(const MinGruParams& p, int r0, int ch) {
  if (ch >= p.width) return;
  T* out = reinterpret_cast<T*>(p.out);
  const T* z = reinterpret_cast<const T*>(p.z) + ch;
  const T* x = reinterpret_cast<const T*>(p.x) + ch;
  const T* g = reinterpret_cast<const T*>(p.g) + ch;
  const int before = max(r0 - 1, 0), behind = min(r0 + 1, p.rows - 1);
  const int64_t slot = p.slots[r0], slot_before = p.slots[before];
  int64_t slot_next = p.slots[behind];
  const int seq = p.seq_ids[r0], seq_before = p.seq_ids[before], pos = p.positions[r0];
  int seq_next = p.seq_ids[behind];
  T zv = z[(size_t)r0 * p.ld], xv = x[(size_t)r0 * p.ld], gv = g[(size_t)r0 * p.ld];
  const float zb = p.zb ? p.zb[ch] : 0.f, xb = p.xb ? p.xb[ch] : 0.f;
  asm volatile("" ::: "memory");  // (all of them ahead of the first decision)
  if (slot < 0) {  // inert row of a padded step
    stv(out + (size_t)r0 * p.ldo + ch, 0.f);
    return;
  }
  if (r0 > 0 && seq_before == seq && slot_before >= 0) return;  // not the head of its run
  float* st = p.state + (size_t)seq * p.state_ld + ch;
  float S = pos > 0 ? *st : 0.f;
  for (int r = r0;;) {
    const Gate gt = min_gru_gate(ldv(&zv) + zb, ldv(&xv) + xb);
    S = min_gru_step(gt, S);
    stv(out + (size_t)r * p.ldo + ch, S * silu(ldv(&gv)) * p.out_scale);
    if (++r == p.rows || seq_next != seq || slot_next < 0) break;
    const size_t o = (size_t)r * p.ld;
    zv = z[o];
    xv = x[o];
    gv = g[o];
    if (r + 1 < p.rows) {
      seq_next = p.seq_ids[r + 1];
      slot_next = p.slots[r + 1];
    }
  }
  *st = S;
}

}  // namespace
