// stm_pairs.hpp — which part of a scan output area a batch wrote.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace stm {

struct ScanOp {
  uint64_t op;   // its index in the batch
  uint64_t len;  // the pairs it asks for: its slots of the output area
};

// The scans' slots lie one after the other, and scan s wrote the first out_vals[s.op] of its own
// (all of them unless the key space ends before): the rest are not the batch's, and what its
// device buffer holds there is another batch's.  Calls f(first, pairs) for every stretch of
// written slots.
template <typename F>
void written_pairs(const ScanOp* scans, size_t n, const uint64_t* out_vals, F&& f) {
  uint64_t from = 0, at = 0;
  for (size_t q = 0; q < n; ++q) {
    const uint64_t wrote = std::min(out_vals[scans[q].op], scans[q].len);
    if (wrote < scans[q].len) {
      if (at + wrote > from) f(from, at + wrote - from);
      from = at + scans[q].len;
    }
    at += scans[q].len;
  }
  if (at > from) f(from, at - from);
}

}  // namespace stm
