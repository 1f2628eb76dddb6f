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
  uint32_t m;    // first INSERTs of a group in the range, as if no group reached in from before it
                 // (bits 0..30); ACC_LEAD: one of them precedes the range's first head
};
constexpr uint32_t ACC_LEAD = 1u << 31;

STM_DEV Acc acc_identity() { return Acc{0u, -1, -1, 0u}; }
// Whether the group the range ends in (open to its right) has an INSERT in the range.
STM_DEV bool acc_open_insert(const Acc& a) { return a.ins >= 0 && a.ins >= a.head; }
STM_DEV Acc acc_combine(const Acc& a, const Acc& b) {
  const uint32_t again = (b.m & ACC_LEAD) && acc_open_insert(a) ? 1u : 0u;
  const uint32_t lead = (a.m | (a.head < 0 ? b.m : 0u)) & ACC_LEAD;
  return Acc{a.c + b.c, max(a.head, b.head), max(a.ins, b.ins),
             ((a.m & ~ACC_LEAD) + (b.m & ~ACC_LEAD) - again) | lead};
}

// Position of the highest lane set in m within a round starting at rb, or `none`.
STM_DEV int32_t last_set(uint64_t m, uint32_t rb, int32_t none) {
  return m ? (int32_t)(rb + 63u - (uint32_t)__clzll((long long)m)) : none;
}

// The lanes of a 64-element round that hold the first INSERT of their group, from the round's
// heads and INSERTs; open: an INSERT of the group that reaches into the round lies before it.
// A lane is not first when an INSERT lies below it with no head in between: s marks the lanes just
// above an INSERT that start no group, and adding s to the non-head lanes p carries each mark up to
// the next head (the bits the sum clears).
STM_DEV uint64_t first_inserts(uint64_t heads, uint64_t ins, bool open) {
  const uint64_t p = ~heads;
  const uint64_t s = ((ins << 1) | (open ? 1ull : 0ull)) & p;
  return ins & ~((((p + s) ^ p) | s) & p);
}

// The state after a round that starts at position rb, from the state before it.
STM_DEV Acc acc_round(const Acc& a, uint64_t heads, uint64_t ins, uint32_t rb) {
  const uint64_t first = first_inserts(heads, ins, acc_open_insert(a));
  const uint64_t lead = heads ? first & ((heads & (0 - heads)) - 1) : first;
  return Acc{a.c + (uint32_t)__popcll(heads), last_set(heads, rb, a.head), last_set(ins, rb, a.ins),
             (a.m + (uint32_t)__popcll(first)) | (lead && a.head < 0 ? ACC_LEAD : 0u)};
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
