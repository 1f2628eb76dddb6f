// stm_scan.hip — range scans with exact sequential semantics inside a batch.
//
// No reference counterpart: the reference declares RANGE (op 3, src/input-helper.h:14-17)
// but never implements it (src/tree.h:37-39, src/main.cpp:30-34), and its v38 leaves keep no
// sibling links (src/gpu-stm-tree-v38/bpt-gpustm-kernel-tree.cuh:413-445).  The v35 variant
// maintains right-sibling pointers on split (src/gpu-stm-tree-v35/bpt-gpustm-kernel-tx.cuh:436-444);
// this tree keeps them in NodeMeta::next.
//
// SCAN(k, L) at input position i returns the first L pairs (x, v) with x >= k in the state
// before op i.  That state is the tree before the batch plus the batch's inserts at input
// positions < i.  Scans therefore run after the per-key fold and before the upsert kernel:
//   * the tree part is read from the unmodified pre-batch tree (leaf, then right siblings; where the
//     batch inserts nothing, the leaves a level-1 node lists, without the merge);
//   * the batch part is read from the fold's output, one group per unique key in key order:
//     a group contributes key x iff its first insert precedes i; its value is the latest
//     insert of x before i, found by a binary search over the group's input positions
//     (stable sort keeps them increasing) and the fold's per-entry "latest insert" index.
// One wavefront merges the two sorted streams 64 candidates at a time: each round takes the
// next leaf chunk and the next 64 groups, finalises every candidate not above the smaller of
// the two chunks' last keys (batch values shadow equal tree keys), places each by its merge
// rank (lane binary searches over the other chunk) and writes up to L - written pairs.
//
// Output layout: scan op i's pairs start at off_i = the sum of L over the scan ops before it
// in input order (three kernels compute off_i); out_vals[i] = pairs written, out_found[i] =
// (pairs > 0), written after the upsert kernel (which answers every non-insert op of a key
// group, scans included, with the key's value).
#include <algorithm>

#include "stm_common.hpp"
#include "stm_internal.hpp"
#include "stm_tree.hpp"

namespace stm {

constexpr int OFF_BLOCK = 256;
constexpr int OFF_ITEMS = 16;
constexpr int OFF_TILE = OFF_BLOCK * OFF_ITEMS;
constexpr uint32_t OFF_SUM_TILES = 1024;
constexpr uint32_t SCAN_GRID_CAP = 2048;
// Wavefronts that share the scans of one 64-op window: at least SCAN_SPLIT, and up to one per scan
// while the batch is too short to give the device SCAN_WAVES wavefronts otherwise; a batch still
// shorter (below 8192 ops) gives every scan SCAN_PARTS of them.  A scan is a chain of round trips, so
// a window holding several scans, or one long scan, sets the kernel's time when few wavefronts run
// them.  4099 ops, half of them scans of 500..8000 pairs, µs a call: 3910 with four wavefronts per window
// and the sibling links, 317 with a wavefront per scan, 196 with whole nodes at a time (scan_plain),
// 157 with four wavefronts per scan.
constexpr uint32_t SCAN_SPLIT = 4;
constexpr uint32_t SCAN_WAVES = 8192;
constexpr uint32_t SCAN_PARTS = 4;
constexpr uint32_t SCAN_ROUND_CAP = 1u << 24;

STM_DEV uint64_t scan_len(uint8_t op, uint64_t v) {
  return (op == OP_RANGE && v >= 1 && v <= SCAN_MAX_LEN) ? v : 0;
}

STM_DEV uint64_t block_exclusive_sum_u64(uint64_t v, uint64_t* s_w /*[4]*/, uint64_t& total) {
  const int lane = lane_id();
  const int wave = threadIdx.x / WAVE;
  uint64_t x = v;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const uint64_t y = shfl64(x, lane - off < 0 ? lane : lane - off);
    if (lane >= off) x += y;
  }
  if (lane == WAVE - 1) s_w[wave] = x;
  __syncthreads();
  uint64_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < OFF_BLOCK / WAVE; ++w) {
    const uint64_t t = s_w[w];
    if (w < wave) before += t;
    total += t;
  }
  __syncthreads();
  return before + x - v;
}

struct ScanIn {
  const uint64_t* keys;
  const uint64_t* vals;
  const uint8_t* ops;
  uint32_t n;
  uint64_t* out_vals;
  uint8_t* out_found;
  uint64_t* scan_keys;
  uint64_t* scan_vals;
  uint64_t scan_cap;
};

STM_DEV ScanIn scan_in(const ScanArgs& a) {
  const BatchDesc* d = a.desc;
  if (d) return ScanIn{d->keys, d->vals, d->ops, d->n, d->out_vals, d->out_found, d->scan_keys,
                       d->scan_vals, d->scan_cap};
  return ScanIn{a.keys, a.vals, a.ops, a.n, a.out_vals, a.out_found, a.scan_keys, a.scan_vals,
                a.scan_cap};
}

// The scan lengths (0 for other ops) of a thread's OFF_ITEMS consecutive ops of tile b, and a bit
// per scan op: every op code in one round of loads (indexes clamped into the batch), then every
// length, instead of a dependent pair of loads per op.
STM_DEV uint32_t load_lengths(const ScanIn& in, uint32_t b, uint64_t (&len)[OFF_ITEMS]) {
  const uint64_t i0 = (uint64_t)b * OFF_TILE + (uint64_t)threadIdx.x * OFF_ITEMS;
  uint8_t op[OFF_ITEMS];
#pragma unroll
  for (int r = 0; r < OFF_ITEMS; ++r) op[r] = in.ops[min(i0 + r, (uint64_t)in.n - 1)];
  uint32_t scans = 0;
#pragma unroll
  for (int r = 0; r < OFF_ITEMS; ++r) {
    const bool is = i0 + r < in.n && op[r] == OP_RANGE;
    len[r] = is ? in.vals[i0 + r] : 0;
    scans |= is ? 1u << r : 0u;
  }
#pragma unroll
  for (int r = 0; r < OFF_ITEMS; ++r) len[r] = (scans >> r) & 1u ? scan_len(OP_RANGE, len[r]) : 0;
  return scans;
}

// Tile sums of the scan lengths in input order.
__global__ __launch_bounds__(OFF_BLOCK) void k_scanoff_reduce(ScanArgs a) {
  __shared__ uint64_t s_w[OFF_BLOCK / WAVE];
  const ScanIn in = scan_in(a);
  const uint32_t ntiles = (in.n + OFF_TILE - 1) / OFF_TILE;
  for (uint32_t b = blockIdx.x; b < ntiles; b += gridDim.x) {
    uint64_t len[OFF_ITEMS];
    (void)load_lengths(in, b, len);
    uint64_t acc = 0;
#pragma unroll
    for (int r = 0; r < OFF_ITEMS; ++r) acc += len[r];
    uint64_t total;
    (void)block_exclusive_sum_u64(acc, s_w, total);
    if (threadIdx.x == 0) a.tile_sums[b] = total;
  }
}

// Exclusive scan of the tile sums (one block); the batch total goes to the counters.  Batches of
// more than OFF_SUM_TILES tiles only: up to there k_scanoff_apply sums the tiles before its own
// itself, at most four loads per thread, which spares a launch.
__global__ __launch_bounds__(OFF_BLOCK) void k_scanoff_tiles(ScanArgs a) {
  __shared__ uint64_t s_w[OFF_BLOCK / WAVE];
  const ScanIn in = scan_in(a);
  const uint32_t ntiles = (in.n + OFF_TILE - 1) / OFF_TILE;
  const uint32_t per = (ntiles + OFF_BLOCK - 1) / OFF_BLOCK;
  const uint32_t b0 = min(threadIdx.x * per, ntiles);
  const uint32_t b1 = min(b0 + per, ntiles);
  uint64_t s = 0;
  for (uint32_t b = b0; b < b1; ++b) s += a.tile_sums[b];
  uint64_t total;
  uint64_t run = block_exclusive_sum_u64(s, s_w, total);
  for (uint32_t b = b0; b < b1; ++b) {
    const uint64_t t = a.tile_sums[b];
    a.tile_sums[b] = run;
    run += t;
  }
  if (threadIdx.x == 0) {
    a.counters->scan_total = total;
    a.counters->scan_bad = 0;
  }
}

// off_i for every scan op (input order), into soff[i].  scanned: tile_sums hold the prefixes
// already (k_scanoff_tiles).  A tile's offsets need two round trips of loads and one scan over the
// block; one scan per 256 ops, each behind its own loads, took 16 µs where this takes 5.
__global__ __launch_bounds__(OFF_BLOCK) void k_scanoff_apply(ScanArgs a, int scanned) {
  __shared__ uint64_t s_w[OFF_BLOCK / WAVE];
  const ScanIn in = scan_in(a);
  const uint32_t ntiles = (in.n + OFF_TILE - 1) / OFF_TILE;
  for (uint32_t b = blockIdx.x; b < ntiles; b += gridDim.x) {
    uint64_t len[OFF_ITEMS];
    const uint32_t scans = load_lengths(in, b, len);
    uint64_t base = 0;
    if (scanned) {
      base = a.tile_sums[b];
    } else {
      uint64_t before = 0;
      for (uint32_t q = threadIdx.x; q < b; q += OFF_BLOCK) before += a.tile_sums[q];
      (void)block_exclusive_sum_u64(before, s_w, base);
    }
    uint64_t acc = 0;
#pragma unroll
    for (int r = 0; r < OFF_ITEMS; ++r) acc += len[r];
    uint64_t total;
    uint64_t at = base + block_exclusive_sum_u64(acc, s_w, total);
    const uint64_t i0 = (uint64_t)b * OFF_TILE + (uint64_t)threadIdx.x * OFF_ITEMS;
#pragma unroll
    for (int r = 0; r < OFF_ITEMS; ++r) {
      if ((scans >> r) & 1u) a.soff[i0 + r] = at;
      at += len[r];
    }
    if (!scanned && b + 1 == ntiles && threadIdx.x == 0) {
      a.counters->scan_total = base + total;
      a.counters->scan_bad = 0;
    }
  }
}

// Number of lanes j < n whose (ascending) value v_j is below x; every lane runs the same
// steps, so the shuffles never read from an inactive lane.
STM_DEV uint32_t lanes_below(uint64_t v, uint32_t n, uint64_t x) {
  uint32_t pos = 0;
#pragma unroll
  for (int step = 64; step >= 1; step >>= 1) {
    const uint32_t probe = min(pos + (uint32_t)step - 1, 63u);
    const uint64_t pv = shfl64(v, (int)probe);
    if (pos + (uint32_t)step <= n && pv < x) pos += step;
  }
  return pos;
}

STM_DEV uint64_t mask_below(uint32_t r) { return r >= 64 ? ~0ull : ((1ull << r) - 1); }

// The children of a level-1 node: child j * WAVE + lane and its separator in id[j], sep[j].
template <int F>
struct Kids {
  static constexpr int SPL = (F + WAVE - 1) / WAVE;
  uint64_t sep[SPL];
  uint32_t id[SPL];
  uint32_t n;     // children
  uint32_t at;    // the one the scan goes on with
  uint32_t up;    // the level-1 node after this one (NODE_NONE: none)
  uint64_t high;  // the node's high fence
};

// Element at (uniform, below F) of a lane-distributed array.
template <int F>
STM_DEV uint32_t lane_at(const uint32_t (&x)[(F + WAVE - 1) / WAVE], uint32_t at) {
  uint32_t r = 0;
#pragma unroll
  for (int j = 0; j < (F + WAVE - 1) / WAVE; ++j)
    if ((at >> 6) == (uint32_t)j) r = (uint32_t)__builtin_amdgcn_readlane((int)x[j], (int)(at & 63));
  return r;
}

template <int F>
STM_DEV void load_kids(const TreeView& t, uint32_t node, Kids<F>& kids) {
  const int lane = lane_id();
#pragma unroll
  for (int j = 0; j < Kids<F>::SPL; ++j) {
    const uint64_t at = (uint64_t)node * F + (uint32_t)min(j * WAVE + lane, F - 1);
    kids.sep[j] = t.keys[at];
    kids.id[j] = (uint32_t)t.vals[at];
  }
  const NodeMeta* m = t.meta + node;
  const uint64_t info = uniform64(m->info), next = uniform64(m->next);
  kids.high = uniform64(m->high);
  kids.n = min(meta_count(info), (uint32_t)F);
  kids.at = 0;
  kids.up = next < t.capacity ? (uint32_t)next : NODE_NONE;
}

// The level-1 node whose child kids.at holds key, by a root-to-leaf descent (each level one round
// trip: a node's keys, children and metadata are loaded together).  A root that is a leaf is its
// own only child.
template <int F>
STM_DEV void wave_find_kids(const TreeView& t, uint64_t key, Kids<F>& kids) {
  const uint32_t cap = t.capacity;
  uint32_t node = (uint32_t)min<uint64_t>(uniform64(t.hdr->root), cap - 1);
  const uint32_t height = (uint32_t)min<uint64_t>(uniform64(t.hdr->height), 64);
  const int lane = lane_id();
#pragma unroll
  for (int j = 0; j < Kids<F>::SPL; ++j) {
    kids.sep[j] = 0;
    kids.id[j] = node;
  }
  kids.n = 1;
  kids.at = 0;
  kids.up = NODE_NONE;
  kids.high = KEY_EMPTY;
  for (uint32_t lvl = height; lvl > 1; --lvl) {
    load_kids<F>(t, node, kids);
    uint32_t cnt = 0;
#pragma unroll
    for (int j = 0; j < Kids<F>::SPL; ++j)
      cnt += (uint32_t)__popcll(ballot(j * WAVE + lane < F && kids.sep[j] <= key));
    kids.at = cnt ? cnt - 1 : 0;
    node = min(lane_at<F>(kids.id, kids.at), cap - 1);
  }
}

// First of the n ascending keys that is not below x: every lane probes one key of the range per
// step, so a step cuts the range 64-fold (three round trips for 2^18 keys).
STM_DEV uint32_t wave_lower_bound(const uint64_t* __restrict__ keys, uint32_t n, uint64_t x) {
  const uint32_t lane = (uint32_t)lane_id();
  uint32_t lo = 0, hi = n;
  while (hi - lo > (uint32_t)WAVE) {
    const uint32_t step = (hi - lo + WAVE - 1) / WAVE;
    const uint32_t at = lo + lane * step;
    const uint32_t below = (uint32_t)__popcll(ballot(at < hi && keys[min(at, n - 1)] < x));
    if (below == 0) return lo;
    const uint32_t up = min(hi, lo + below * step);
    lo += (below - 1) * step + 1;
    hi = up;
  }
  const uint32_t at = lo + lane;
  return lo + (n ? (uint32_t)__popcll(ballot(at < hi && keys[min(at, n - 1)] < x)) : 0u);
}

// A leaf in registers: slot j * WAVE + lane of its keys and values.  Free slots hold KEY_EMPTY, so
// the entry count need not be known to load it.  As loaded, lanes past a leaf of 32 slots hold its
// last one: a select on a key here would wait for the load (mask_slots does it later).
template <int F>
struct LeafLoad {
  static constexpr int SPL = (F + WAVE - 1) / WAVE;
  uint64_t k[SPL], v[SPL];
};

template <int F>
STM_DEV void load_leaf(const TreeView& t, uint32_t leaf, LeafLoad<F>& b) {
  const int lane = lane_id();
#pragma unroll
  for (int j = 0; j < LeafLoad<F>::SPL; ++j) {
    const uint64_t at = (uint64_t)leaf * F + (uint32_t)min(j * WAVE + lane, F - 1);
    b.k[j] = t.keys[at];
    b.v[j] = t.vals[at];
  }
}

template <int F>
STM_DEV void mask_slots(LeafLoad<F>& b) {
  if constexpr (F < WAVE) b.k[0] = lane_id() < F ? b.k[0] : KEY_EMPTY;
}

// Element p (lane-dependent, p < F) of a leaf held in registers.
template <int F, typename T>
STM_DEV T at_position(const T (&x)[(F + WAVE - 1) / WAVE], uint32_t p) {
  T r = x[0];
#pragma unroll
  for (int j = 0; j < (F + WAVE - 1) / WAVE; ++j) {
    T v;
    if constexpr (sizeof(T) == 8) v = shfl64(x[j], (int)(p & 63));
    else v = (T)__shfl((int)x[j], (int)(p & 63), WAVE);
    if ((p >> 6) == (uint32_t)j) r = v;
  }
  return r;
}

// The entries of a loaded leaf in key order: position j * WAVE + lane holds key b.k[j] and value
// b.v[j] (KEY_EMPTY past the last).  A bulk-built leaf and both halves of a split are in key order
// until an insert is appended, which one comparison with the next slot shows; others go through
// a bitonic sorting network over the wavefront's N = WAVE * SPL elements (element j * WAVE +
// lane in register j): 21 compare-exchange steps for N = 64, 28 for 128, each a lane shuffle of
// the key and slot (or, at distance 64, the lane's other register).  The keys are distinct and
// KEY_EMPTY pads past the last, so the order is exact.  (Ranking each entry with two wave-uniform
// passes over the entries took a serving batch's scan kernel from 49 to 115 µs.)
template <int F>
STM_DEV void leaf_in_key_order(LeafLoad<F>& b) {
  constexpr int SPL = LeafLoad<F>::SPL;
  constexpr uint32_t N = (uint32_t)(WAVE * SPL);
  static_assert(SPL == 1 || SPL == 2, "one or two slots per lane");
  const uint32_t lane = (uint32_t)lane_id();
  bool in_order = true;
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const uint64_t right = shfl64(b.k[j], (int)min(lane + 1, (uint32_t)WAVE - 1));
    uint64_t next = right;
    if constexpr (SPL == 2) {
      const uint64_t first = readlane64(b.k[1], 0);
      next = lane == WAVE - 1 ? (j == 0 ? first : KEY_EMPTY) : right;
    }
    in_order = in_order && b.k[j] <= next;
  }
  if (ballot(!in_order) == 0) return;
  uint64_t (&sk)[SPL] = b.k;
  uint32_t ss[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) ss[j] = (uint32_t)j * WAVE + lane;
#pragma unroll
  for (uint32_t size = 2; size <= N; size <<= 1) {
#pragma unroll
    for (uint32_t d = size >> 1; d > 0; d >>= 1) {
      if (d >= (uint32_t)WAVE) {
        // SPL == 2, d == 64: elements lane and 64 + lane, both in this lane
        if constexpr (SPL == 2) {
          const bool up = (lane & size) == 0;  // ascending block (size >= 128 here)
          const bool sw = up ? sk[1] < sk[0] : sk[0] < sk[1];
          const uint64_t k0 = sk[0];
          const uint32_t s0 = ss[0];
          if (sw) {
            sk[0] = sk[1];
            ss[0] = ss[1];
            sk[1] = k0;
            ss[1] = s0;
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < SPL; ++j) {
          const uint32_t e = (uint32_t)j * WAVE + lane;
          const uint64_t pk = shfl64(sk[j], (int)(lane ^ d));
          const uint32_t ps = (uint32_t)__shfl((int)ss[j], (int)(lane ^ d), WAVE);
          const bool up = (e & size) == 0;
          const bool lower = (e & d) == 0;
          // the lower element of an ascending pair keeps the smaller key, and so on
          const bool take = (lower == up) ? pk < sk[j] : pk > sk[j];
          if (take) {
            sk[j] = pk;
            ss[j] = ps;
          }
        }
      }
    }
  }
  uint64_t sv[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) sv[j] = at_position<F>(b.v, ss[j]);
#pragma unroll
  for (int j = 0; j < SPL; ++j) b.v[j] = sv[j];
}

// Leaves of the fast form read in one round trip, and 64-group windows of the batch it looks
// through for inserts before it gives up.
template <int F>
constexpr uint32_t scan_chunk() {
  return F > WAVE ? 4 : 8;
}
constexpr uint32_t SCAN_GROUP_WINDOWS = 4;

// A scan over stretches of the tree into which the batch inserts nothing: a level-1 node's leaves
// and their entry counts are known at once, so every leaf's place in the output is too, and the
// leaves are read a chunk at a time (a step along the sibling links, load, order and store, took
// about 1.9 µs a leaf, whatever was loaded ahead).  Goes on from node to node; returns true when the scan is
// complete, false when a node's stretch meets an insert (kids.at: the leaf to go on with; first: it
// is still the leaf of k).  Of PARTS wavefronts that run the scan, the part-th takes every PARTS-th
// chunk.
template <int F, uint32_t PARTS>
STM_DEV bool scan_plain(const TreeView& t, const ScanArgs& a, const ScanIn& in, uint32_t U, uint64_t k,
                        uint32_t L, uint64_t off, uint32_t part, Kids<F>& kids,
                        uint32_t& bg, uint32_t& cnt, bool& first) {
  constexpr int SPL = (F + WAVE - 1) / WAVE;
  constexpr uint32_t C = scan_chunk<F>();
  const uint32_t lane = (uint32_t)lane_id();
  const uint32_t cap = t.capacity;
  uint32_t turn = part;  // chunks until this wavefront's next one
  for (uint32_t node = 0; node < cap; ++node) {
    const uint32_t room = L - cnt;
    const uint32_t avail = kids.n - kids.at;
    LeafLoad<F> b[C];
    auto load_chunk = [&](uint32_t q, uint32_t m) {
#pragma unroll
      for (uint32_t e = 0; e < C; ++e)
        if (q + e < m) load_leaf<F>(t, min(lane_at<F>(kids.id, kids.at + q + e), cap - 1), b[e]);
    };
    // In one round trip: the entry counts of the node's leaves, the first chunk (as many leaves as
    // the scan may take where they are half full), the batch's next groups.
    uint32_t c[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const uint32_t at = (uint32_t)(j * WAVE) + lane;
      const bool v = at >= kids.at && at < kids.n;
      c[j] = v ? meta_count(t.meta[min(kids.id[j], cap - 1)].info) : 0u;
    }
    const uint32_t early = max(min(min(room / (F / 2) + 2, C), avail), 1u);
    load_chunk(0, turn == 0 ? early : first ? 1u : 0u);  // every wavefront looks at k's own leaf
    uint64_t gk = bg + lane < U ? a.ukey[bg + lane] : KEY_EMPTY;
    uint32_t gop = bg + lane < U ? a.uop[bg + lane] : 0u;
    // Entries before each leaf (from kids.at on), and how many leaves the scan needs.
    uint32_t start[SPL], sum = 0;
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      uint32_t x = c[j];
#pragma unroll
      for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, o, WAVE);
        if (lane >= (uint32_t)o) x += y;
      }
      start[j] = sum + x - c[j];
      sum += (uint32_t)__builtin_amdgcn_readlane((int)x, WAVE - 1);
    }
    uint32_t below = 0;  // entries of the first leaf before k
    if (first) {
      mask_slots<F>(b[0]);
#pragma unroll
      for (int j = 0; j < SPL; ++j) below += (uint32_t)__popcll(ballot(b[0].k[j] < k));
    }
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const uint32_t at = (uint32_t)(j * WAVE) + lane;
      m += (uint32_t)__popcll(ballot(at >= kids.at && at < kids.n && start[j] < room + below));
    }
    m = max(m, 1u);
    uint64_t end = kids.high;
    if (kids.at + m < kids.n) {
#pragma unroll
      for (int j = 0; j < SPL; ++j)
        if (((kids.at + m) >> 6) == (uint32_t)j) end = readlane64(kids.sep[j], (int)((kids.at + m) & 63));
    }
    // The groups below the stretch's end: any insert among them ends the fast form.
    uint32_t gw = bg;
    for (uint32_t w = 0;; ++w) {
      const bool inside = gw + lane < U && gk < end;
      if (ballot(inside && gop == OP_INSERT)) return false;
      const uint32_t n = (uint32_t)__popcll(ballot(inside));
      gw += n;
      if (n < (uint32_t)WAVE) break;
      if (w + 1 >= SCAN_GROUP_WINDOWS) return false;
      gk = gw + lane < U ? a.ukey[gw + lane] : KEY_EMPTY;
      gop = gw + lane < U ? a.uop[gw + lane] : 0u;
    }
    uint32_t have = early;  // leaves of the current chunk
    for (uint32_t q = 0; q < m; q += have) {
      if (q > 0) have = C;
      if (turn-- > 0) continue;
      turn = PARTS - 1;
      if (q > 0) load_chunk(q, m);
#pragma unroll
      for (uint32_t e = 0; e < C; ++e) {
        if (e < have && q + e < m) {
          LeafLoad<F>& x = b[e];
          mask_slots<F>(x);
          leaf_in_key_order<F>(x);
          const uint32_t s0 = lane_at<F>(start, kids.at + q + e);
#pragma unroll
          for (int j = 0; j < SPL; ++j) {
            const uint32_t p = s0 + (uint32_t)(j * WAVE) + lane;  // entries from the first leaf's on
            if (x.k[j] != KEY_EMPTY && p >= below && p - below < room) {
              in.scan_keys[off + cnt + (p - below)] = x.k[j];
              in.scan_vals[off + cnt + (p - below)] = x.v[j];
            }
          }
        }
      }
    }
    // Entries of the leaves taken, less those before k.
    const uint32_t held = (kids.at + m < kids.n ? lane_at<F>(start, kids.at + m) : sum) - below;
    cnt += min(held, room);
    kids.at += m;
    bg = gw;
    if (cnt >= L) return true;
    first = false;
    if (kids.up == NODE_NONE) return true;
    load_kids<F>(t, kids.up, kids);
  }
  return true;
}

// One scan op, run by the whole wavefront; returns the pairs written.  Where the batch inserts into
// its range the leaf chain is walked along the sibling links instead, merged with the batch.
template <int F, uint32_t PARTS>
STM_DEV uint32_t run_scan(const TreeView& t, const ScanArgs& a, const ScanIn& in, uint32_t U,
                          uint64_t k, uint32_t i, uint32_t L, uint64_t off, uint32_t part) {
  const int lane = lane_id();
  const uint32_t cap = t.capacity;
  constexpr int SPL = (F + WAVE - 1) / WAVE;
  Kids<F> kids;
  wave_find_kids<F>(t, k, kids);
  // First group with key >= k (groups are in ascending key order).
  uint32_t bg = uniform32(wave_lower_bound(a.ukey, U, k));
  uint32_t cnt = 0;
  bool first = true;
  if (scan_plain<F, PARTS>(t, a, in, U, k, L, off, part, kids, bg, cnt, first) || part > 0)
    return cnt;
  LeafLoad<F> cur, ahead;
  uint64_t cur_next, ahead_next = NODE_NONE;
  const uint32_t leaf0 = min(lane_at<F>(kids.id, kids.at), cap - 1);
  load_leaf<F>(t, leaf0, cur);
  cur_next = t.meta[leaf0].next;
  uint32_t tl = NODE_NONE;  // the next leaf of the chain, NODE_NONE at its end
  bool loaded = false;      // `ahead` holds it
  uint32_t ts = 0, tcount = 0;  // key-order positions [ts, tcount) of cur are left
  bool t_done = false;
  // Makes the leaf in `cur` current: its entries into key order, its right sibling under way when
  // the scan will go past it.
  auto enter = [&](uint64_t from) {
    mask_slots<F>(cur);
    const uint64_t nx = uniform64(cur_next);
    tl = nx < cap ? (uint32_t)nx : NODE_NONE;
    tcount = 0;
    ts = 0;
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      tcount += (uint32_t)__popcll(ballot(cur.k[j] != KEY_EMPTY));
      ts += (uint32_t)__popcll(ballot(cur.k[j] < from));
    }
    loaded = tl != NODE_NONE && L - cnt > tcount - ts;
    if (loaded) {
      load_leaf<F>(t, tl, ahead);
      ahead_next = t.meta[tl].next;
    }
    leaf_in_key_order<F>(cur);
  };
  enter(first ? k : 0);
  // The groups [bg, bg + 64) as the scan sees them, loaded when bg moves: key, whether the group
  // inserts before op i, and the value it then holds.
  uint32_t bn = 0, bg_at = NODE_NONE;
  uint64_t bk = KEY_EMPTY, bval = 0;
  bool bv = false, vis = false;
  // Every round consumes a whole chunk of one stream; the caps only guard a corrupt pool.
  for (uint32_t round = 0; cnt < L && round < SCAN_ROUND_CAP; ++round) {
    // Next non-empty leaf chunk.
    for (uint32_t hop = 0; !t_done && ts >= tcount; ++hop) {
      if (tl == NODE_NONE || hop >= SCAN_ROUND_CAP) {
        t_done = true;
      } else {
        if (!loaded) {
          load_leaf<F>(t, tl, ahead);
          ahead_next = t.meta[tl].next;
        }
        cur = ahead;
        cur_next = ahead_next;
        enter(0);
      }
    }
    if (t_done && bg >= U) break;
    const uint32_t tn = t_done ? 0u : min(tcount - ts, (uint32_t)WAVE);
    const bool tv = (uint32_t)lane < tn;
    // Key-order position ts + lane, read from every lane (the shuffles need their sources
    // active) and then selected.
    const uint32_t tp = min(ts + (uint32_t)lane, (uint32_t)F - 1);
    const uint64_t tk_at = at_position<F>(cur.k, tp);
    const uint64_t tval = at_position<F>(cur.v, tp);
    const uint64_t tk = tv ? tk_at : KEY_EMPTY;
    const bool t_more = !t_done && (ts + tn < tcount || tl != NODE_NONE);
    const uint64_t lastT = t_more ? readlane64(tk, (int)tn - 1) : KEY_EMPTY;

    if (bg != bg_at) {
      bg_at = bg;
      bn = bg < U ? min(U - bg, (uint32_t)WAVE) : 0u;
      bv = (uint32_t)lane < bn;
      bk = KEY_EMPTY;
      bval = 0;
      vis = false;
      if (bv) {
        const uint32_t g = bg + lane;
        bk = a.ukey[g];
        if (a.uop[g] == OP_INSERT) {
          const uint32_t gs = a.gstart[g];
          const uint32_t fi = gs + max(a.npend[g], 1u) - 1;  // sorted index of the first insert
          const uint32_t ge = (g + 1 < U) ? a.gstart[g + 1] : in.n;
          if (pos_of(a.sidx[fi]) < i) {
            uint32_t lo = fi, hi = ge;  // sidx[lo] < i; the last such entry lies in [lo, hi)
            while (hi - lo > 1) {
              const uint32_t mid = (lo + hi) >> 1;
              if (pos_of(a.sidx[mid]) < i) lo = mid;
              else hi = mid;
            }
            const int32_t li = a.lastins[lo];
            if (li >= 0) {
              vis = true;
              bval = in.vals[pos_of(a.sidx[li])];
            }
          }
        }
      }
    }
    const uint32_t room = L - cnt;
    if (tn && (bn == 0 || readlane64(bk, 0) > lastT)) {
      // No group of the batch falls into this chunk: its entries as they are.
      if (tv && (uint32_t)lane < room) {
        in.scan_keys[off + cnt + lane] = tk;
        in.scan_vals[off + cnt + lane] = tval;
      }
      cnt += min(tn, room);
      ts += tn;
      continue;
    }
    const bool b_more = bg + bn < U;
    const uint64_t lastB = b_more ? readlane64(bk, (int)bn - 1) : KEY_EMPTY;
    const uint64_t bound = min(lastT, lastB);

    const bool t_el = tv && tk <= bound;
    const bool b_raw = bv && bk <= bound;
    const bool b_el = b_raw && vis;
    const uint64_t visM = ballot(b_el);
    const uint32_t rB = lanes_below(bk, bn, tk);  // groups below this tree key
    const uint64_t bk_at = shfl64(bk, (int)min(rB, 63u));
    const bool shadow = t_el && rB < bn && bk_at == tk && ((visM >> rB) & 1ull);
    const uint64_t shM = ballot(shadow);
    const uint64_t tM = ballot(t_el);
    const uint32_t rT = lanes_below(tk, tn, bk);  // tree keys below this group key
    const uint64_t lt = lanemask_lt();
    if (t_el && !shadow) {
      const uint32_t p = (uint32_t)lane - (uint32_t)__popcll(shM & lt) +
                         (uint32_t)__popcll(visM & mask_below(rB));
      if (p < room) {
        in.scan_keys[off + cnt + p] = tk;
        in.scan_vals[off + cnt + p] = tval;
      }
    }
    if (b_el) {
      const uint32_t p = (uint32_t)__popcll(visM & lt) + rT - (uint32_t)__popcll(shM & mask_below(rT));
      if (p < room) {
        in.scan_keys[off + cnt + p] = bk;
        in.scan_vals[off + cnt + p] = bval;
      }
    }
    const uint32_t emitted = (uint32_t)(__popcll(tM) - __popcll(shM) + __popcll(visM));
    cnt += min(emitted, room);
    ts += (uint32_t)__popcll(tM);
    bg += (uint32_t)__popcll(ballot(b_raw));
  }
  return cnt;
}

// One wavefront per window of 64 input positions: the window's scan ops run one after the
// other, each by the whole wavefront.  soff[i] gets the pair count of scan op i in its upper bits
// (another part's wavefront may read the offset after that; it is below 2^47: 2^30 ops of 2^16 pairs).
constexpr int SCAN_OFF_BITS = 47;
template <int F, uint32_t PARTS>
__global__ __launch_bounds__(256) void k_range_scan(TreeView t, ScanArgs a, uint32_t split) {
  const ScanIn in = scan_in(a);
  const uint32_t U = a.counters->n_unique;
  const int lane = lane_id();
  const uint64_t wave0 = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = (uint64_t)gridDim.x * blockDim.x / WAVE;
  const uint64_t nwin = ((uint64_t)in.n + WAVE - 1) / WAVE;
  const uint64_t lt = lanemask_lt();
  // Work item p = (window, share, part): the wavefront runs the scans of the window
  // whose rank among the window's scans is its share modulo split, so a window with several scans
  // spreads them over split wavefronts.
  for (uint64_t p = wave0; p < nwin * split * PARTS; p += nwaves) {
    const uint32_t part = (uint32_t)(p % PARTS);
    const uint64_t w = p / PARTS / split;
    const uint32_t share = (uint32_t)(p / PARTS % split);
    const uint64_t i_l = w * WAVE + lane;
    const bool is_scan = i_l < in.n && in.ops[i_l] == OP_RANGE;
    const uint32_t rank = (uint32_t)__popcll(ballot(is_scan) & lt);
    const bool mine = is_scan && rank % split == share;
    uint64_t todo = ballot(mine);
    uint64_t k_l = 0, v_l = 0, off_l = 0;
    if (mine) {
      k_l = in.keys[i_l];
      v_l = in.vals[i_l];
      off_l = a.soff[i_l] & ((1ull << SCAN_OFF_BITS) - 1);
    }
    while (todo) {
      const int src = __builtin_ctzll(todo);
      todo &= todo - 1;
      const uint64_t k = readlane64(k_l, src);
      const uint64_t L = readlane64(v_l, src);
      const uint64_t off = readlane64(off_l, src);
      const uint32_t i = (uint32_t)(w * WAVE + src);
      uint32_t c = 0;
      const bool ok = L >= 1 && L <= SCAN_MAX_LEN && off + L <= in.scan_cap && k != KEY_EMPTY;
      if (ok) {
        c = run_scan<F, PARTS>(t, a, in, U, k, i, (uint32_t)L, off, part);
      } else if (lane == 0 && part == 0) {
        atomicAdd(&a.counters->scan_bad, 1u);
      }
      if (lane == src && part == 0) a.soff[i_l] = off | ((uint64_t)c << SCAN_OFF_BITS);
    }
  }
}

// After the upsert kernel: the scan ops' answers.
__global__ __launch_bounds__(256) void k_scan_answers(ScanArgs a) {
  const ScanIn in = scan_in(a);
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < in.n; i += (uint64_t)gridDim.x * 256ull) {
    if (in.ops[i] == OP_RANGE) {
      const uint64_t c = a.soff[i] >> SCAN_OFF_BITS;
      in.out_vals[i] = c;
      in.out_found[i] = c ? 1 : 0;
    }
  }
}

size_t scan_tile_words(uint64_t n) {
  uint64_t t = (n + OFF_TILE - 1) / OFF_TILE;
  return (size_t)std::max<uint64_t>(t, 1);
}

hipError_t launch_scan_offsets(const ScanArgs& a, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  const uint32_t ntiles = (a.n + OFF_TILE - 1) / OFF_TILE;
  const uint32_t grid = std::min<uint32_t>(ntiles, SCAN_GRID_CAP);
  k_scanoff_reduce<<<grid, OFF_BLOCK, 0, s>>>(a);
  const int scanned = ntiles > OFF_SUM_TILES ? 1 : 0;
  if (scanned) k_scanoff_tiles<<<1, OFF_BLOCK, 0, s>>>(a);
  k_scanoff_apply<<<grid, OFF_BLOCK, 0, s>>>(a, scanned);
  return hipGetLastError();
}

template <int F>
static hipError_t launch_range_scan_f(const TreeView& t, const ScanArgs& a, hipStream_t s) {
  const uint64_t windows = ((uint64_t)a.n + WAVE - 1) / WAVE;
  uint32_t split = SCAN_SPLIT;
  while (split < (uint32_t)WAVE && windows * split < SCAN_WAVES) split *= 2;
  const bool parts = split == (uint32_t)WAVE && windows * split < SCAN_WAVES;
  const uint64_t waves = windows * split * (parts ? SCAN_PARTS : 1u);
  const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((waves + 3) / 4, SCAN_WAVES));
  if (parts) k_range_scan<F, SCAN_PARTS><<<blocks, 256, 0, s>>>(t, a, split);
  else k_range_scan<F, 1><<<blocks, 256, 0, s>>>(t, a, split);
  return hipGetLastError();
}

hipError_t launch_range_scan(const TreeView& t, const ScanArgs& a, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  switch (t.fanout) {
    case 32: return launch_range_scan_f<32>(t, a, s);
    case 64: return launch_range_scan_f<64>(t, a, s);
    case 128: return launch_range_scan_f<128>(t, a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_scan_answers(const ScanArgs& a, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(((uint64_t)a.n + 255) / 256, 4096));
  k_scan_answers<<<blocks, 256, 0, s>>>(a);
  return hipGetLastError();
}

}  // namespace stm
