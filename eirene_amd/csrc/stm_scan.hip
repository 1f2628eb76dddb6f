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
//   * the tree part is read from the unmodified pre-batch tree (leaf, then right siblings);
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
// while the batch is too short to give the device SCAN_WAVES wavefronts otherwise.  A scan is a
// chain of dependent leaf reads, so a window holding several scans sets the kernel's time when
// few wavefronts run them all (4099 ops, half of them scans of 500..8000 pairs: 3.91 ms a call
// with four wavefronts per window and no load ahead, 0.41 ms now).
constexpr uint32_t SCAN_SPLIT = 4;
constexpr uint32_t SCAN_WAVES = 8192;
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

// The leaf that holds key, by a root-to-leaf descent (each level one round trip: a node's keys and
// children are loaded together).
template <int F>
STM_DEV uint32_t wave_find_leaf(const TreeView& t, uint64_t key) {
  constexpr int SPL = (F + WAVE - 1) / WAVE;
  const uint32_t cap = t.capacity;
  uint32_t node = (uint32_t)min<uint64_t>(uniform64(t.hdr->root), cap - 1);
  const uint32_t height = (uint32_t)min<uint64_t>(uniform64(t.hdr->height), 64);
  const int lane = lane_id();
  for (uint32_t lvl = height; lvl > 1; --lvl) {
    uint64_t k[SPL], v[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const uint64_t at = (uint64_t)node * F + (uint32_t)min(j * WAVE + lane, F - 1);
      k[j] = t.keys[at];
      v[j] = t.vals[at];
    }
    uint32_t cnt = 0;
#pragma unroll
    for (int j = 0; j < SPL; ++j)
      cnt += (uint32_t)__popcll(ballot(j * WAVE + lane < F && k[j] <= key));
    const uint32_t slot = cnt ? cnt - 1 : 0;
    uint64_t child = 0;
#pragma unroll
    for (int j = 0; j < SPL; ++j)
      if ((slot >> 6) == (uint32_t)j) child = readlane64(v[j], (int)(slot & 63));
    node = (uint32_t)min<uint64_t>(child, cap - 1);
  }
  return node;
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

// A leaf on its way into registers: slot j * WAVE + lane of its keys and values, and its right
// sibling.  Free slots hold KEY_EMPTY, so the entry count need not be known to load it.
template <int F>
struct LeafLoad {
  static constexpr int SPL = (F + WAVE - 1) / WAVE;
  uint64_t k[SPL], v[SPL];
  uint64_t next;
};

template <int F>
STM_DEV void load_leaf(const TreeView& t, uint32_t leaf, LeafLoad<F>& b) {
  const int lane = lane_id();
  b.next = t.meta[leaf].next;
#pragma unroll
  for (int j = 0; j < LeafLoad<F>::SPL; ++j) {
    const int sl = j * WAVE + lane;
    const uint64_t at = (uint64_t)leaf * F + (uint32_t)min(sl, F - 1);
    const uint64_t k = t.keys[at];
    b.v[j] = t.vals[at];
    b.k[j] = sl < F ? k : KEY_EMPTY;
  }
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

// One scan op, run by the whole wavefront; returns the pairs written.  The leaf chain is walked one
// leaf ahead: the right sibling's load goes out before the current leaf is ordered and written, so
// a step costs the longer of the two instead of their sum.  Bound by that chain's latency (about
// 1 µs a leaf), not by bytes.
template <int F>
STM_DEV uint32_t run_scan(const TreeView& t, const ScanArgs& a, const ScanIn& in, uint32_t U,
                          uint64_t k, uint32_t i, uint32_t L, uint64_t off) {
  const int lane = lane_id();
  const uint32_t cap = t.capacity;
  constexpr int SPL = (F + WAVE - 1) / WAVE;
  LeafLoad<F> cur, ahead;
  load_leaf<F>(t, wave_find_leaf<F>(t, k), cur);
  // First group with key >= k (groups are in ascending key order).
  uint32_t bg = wave_lower_bound(a.ukey, U, k);
  uint32_t cnt = 0;
  uint32_t tl = NODE_NONE;  // the next leaf of the chain, NODE_NONE at its end
  bool loaded = false;      // `ahead` holds it
  uint32_t ts = 0, tcount = 0;  // key-order positions [ts, tcount) of cur are left
  bool t_done = false;
  // Makes the leaf in `cur` current: its entries into key order, its right sibling under way when
  // the scan will go past it.
  auto enter = [&](uint64_t from) {
    const uint64_t nx = uniform64(cur.next);
    tl = nx < cap ? (uint32_t)nx : NODE_NONE;
    tcount = 0;
    ts = 0;
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      tcount += (uint32_t)__popcll(ballot(cur.k[j] != KEY_EMPTY));
      ts += (uint32_t)__popcll(ballot(cur.k[j] < from));
    }
    loaded = tl != NODE_NONE && L - cnt > tcount - ts;
    if (loaded) load_leaf<F>(t, tl, ahead);
    leaf_in_key_order<F>(cur);
  };
  enter(k);
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
        if (!loaded) load_leaf<F>(t, tl, ahead);
        cur = ahead;
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
// other, each by the whole wavefront.  soff[i] becomes the pair count of scan op i.
template <int F>
__global__ __launch_bounds__(256) void k_range_scan(TreeView t, ScanArgs a, uint32_t split) {
  const ScanIn in = scan_in(a);
  const uint32_t U = a.counters->n_unique;
  const int lane = lane_id();
  const uint64_t wave0 = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / WAVE;
  const uint64_t nwaves = (uint64_t)gridDim.x * blockDim.x / WAVE;
  const uint64_t nwin = ((uint64_t)in.n + WAVE - 1) / WAVE;
  const uint64_t lt = lanemask_lt();
  // Work item p = (window p / split, share p % split): the wavefront runs the scans of the window
  // whose rank among the window's scans is p % split modulo split, so a window with several scans
  // spreads them over split wavefronts.
  for (uint64_t p = wave0; p < nwin * split; p += nwaves) {
    const uint64_t w = p / split;
    const uint32_t share = (uint32_t)(p % split);
    const uint64_t i_l = w * WAVE + lane;
    const bool is_scan = i_l < in.n && in.ops[i_l] == OP_RANGE;
    const uint32_t rank = (uint32_t)__popcll(ballot(is_scan) & lt);
    const bool mine = is_scan && rank % split == share;
    uint64_t todo = ballot(mine);
    uint64_t k_l = 0, v_l = 0, off_l = 0;
    if (mine) {
      k_l = in.keys[i_l];
      v_l = in.vals[i_l];
      off_l = a.soff[i_l];
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
        c = run_scan<F>(t, a, in, U, k, i, (uint32_t)L, off);
      } else if (lane == 0) {
        atomicAdd(&a.counters->scan_bad, 1u);
      }
      if (lane == src) a.soff[i_l] = c;
    }
  }
}

// After the upsert kernel: the scan ops' answers.
__global__ __launch_bounds__(256) void k_scan_answers(ScanArgs a) {
  const ScanIn in = scan_in(a);
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < in.n; i += (uint64_t)gridDim.x * 256ull) {
    if (in.ops[i] == OP_RANGE) {
      const uint64_t c = a.soff[i];
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
  const uint64_t waves = windows * split;
  const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((waves + 3) / 4, SCAN_GRID_CAP));
  k_range_scan<F><<<blocks, 256, 0, s>>>(t, a, split);
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
