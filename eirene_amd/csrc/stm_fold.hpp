// stm_fold.hpp — device helpers of the per-key fold, shared by the three-kernel fold of large
// batches (stm_fold.hip) and the front half of small ones (stm_front.hip).
#pragma once
#include "stm_common.hpp"
#include "stm_internal.hpp"

namespace stm {

// What the fold needs of a range of the sorted batch.
struct Acc {
  uint32_t c;    // group heads in the range
  int32_t head;  // position of the last head (-1 if none)
  int32_t ins;   // position of the last INSERT (-1 if none)
};

STM_DEV Acc acc_identity() { return Acc{0u, -1, -1}; }
STM_DEV Acc acc_combine(const Acc& a, const Acc& b) {
  return Acc{a.c + b.c, max(a.head, b.head), max(a.ins, b.ins)};
}

// Position of the highest lane set in m within a round starting at rb, or `none`.
STM_DEV int32_t last_set(uint64_t m, uint32_t rb, int32_t none) {
  return m ? (int32_t)(rb + 63u - (uint32_t)__clzll((long long)m)) : none;
}

// With a batch descriptor the element count and the caller's arrays come from device memory
// (one launch sequence serves every batch size).
STM_DEV void fold_resolve(FoldArgs& a) {
  const BatchDesc* d = a.desc;
  if (!d) return;
  a.n = d->n;
  a.vals = d->vals;
  a.ops = d->ops;
  a.out_vals = d->out_vals;
  a.out_found = d->out_found;
}

}  // namespace stm
