// stm_tree.hip — B+tree kernels for gfx950: bottom-up build, read-only batched lookup,
// transactional upsert (STM), dump and structural check.
//
// Reference counterpart: tx_insert_kernel (src/gpu-stm-tree-v38/bpt-gpustm-kernel.cu:15-258)
// with its device library (bpt-gpustm-kernel-tree.cuh, bpt-gpustm-kernel-tx.cuh).  The
// reference runs every unique key of a batch as a transaction on one 32-lane warp.  Here
// the merged ops of a batch are split by type (the merged ops touch distinct keys, so
// they commute):
//   * merged GETs run first in k_lookup on a tree no one writes, walking the sorted keys
//     in chunks with the last inner node and leaf cached in registers;
//   * merged INSERTs then run leaf by leaf: in key order the inserts of a leaf are neighbours, so
//     k_upsert_runs gives each leaf's run to the lanes of one wavefront and k_upsert_long the long
//     ones to a workgroup; leaves that overfill are split there, and k_upsert_parents and
//     k_upsert_finish bring the new nodes to their parents level by level;
//   * what that leaves (a pool that is all but full; every long run when upsert_ops_per_wave asks
//     for less than a wavefront's worth of ops) runs as transactions on 64-lane wavefronts
//     (k_upsert, k_upsert_finish): begin (root + version), optimistic reads validated by fences and
//     lock versions, try-lock commit of the write set with 64-bit CAS, abort and retry with
//     backoff, preemptive split of full inner nodes on the way down
//     (reference: src/gpu-stm-tree-v38/bpt-gpustm-kernel.cu:162-181).
#include <atomic>
#include "stm_common.hpp"
#include "stm_internal.hpp"
#include "stm_learned.hpp"
#include "stm_tree.hpp"

namespace stm {

constexpr uint32_t LOOKUP_GRID_CAP = 8192;
constexpr uint32_t LONG_BLOCKS = 256;        // workgroups of k_upsert_long
constexpr uint32_t PARENT_BLOCKS = 512;      // workgroups of k_upsert_parents
constexpr uint32_t ONE_BLOCK_OPS = 2048;     // batches of at most this many ops upsert in one workgroup
constexpr uint32_t FEW_INSERTS = 1u << 14;   // batches of at most this many ops skip that launch

// ================================================================== bulk build
template <int F>
__global__ void k_build_leaves(TreeView t, const uint64_t* __restrict__ ukey,
                               const uint64_t* __restrict__ uval, uint32_t U, uint32_t fill,
                               uint32_t L, uint64_t* __restrict__ lows_out) {
  const uint64_t gi = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  if (gi >= (uint64_t)L * F) return;
  const uint32_t leaf = (uint32_t)(gi / F);
  const uint32_t s = (uint32_t)(gi % F);
  const uint64_t first = (uint64_t)leaf * fill;
  const uint64_t src = first + s;
  const bool valid = s < fill && src < U;
  t.keys[gi] = valid ? ukey[src] : KEY_EMPTY;
  t.vals[gi] = valid ? uval[src] : 0;
  if (s == 0) {
    const uint32_t cnt = U > first ? (uint32_t)min<uint64_t>(fill, U - first) : 0u;
    NodeMeta m{};
    m.lock = 0;
    m.info = make_info(cnt, 0);
    m.low = leaf == 0 ? 0 : ukey[first];
    m.high = (leaf + 1 < L) ? ukey[first + fill] : KEY_EMPTY;
    m.next = (leaf + 1 < L) ? (uint64_t)(leaf + 1) : (uint64_t)NODE_NONE;
    t.meta[leaf] = m;
    lows_out[leaf] = m.low;
  }
}

template <int F>
__global__ void k_build_inner(TreeView t, const uint64_t* __restrict__ lows_prev, uint32_t n_prev,
                              uint32_t first_prev, uint32_t fill, uint32_t n_this,
                              uint32_t first_this, uint32_t level, uint64_t* __restrict__ lows_out) {
  const uint64_t gi = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  if (gi >= (uint64_t)n_this * F) return;
  const uint32_t j = (uint32_t)(gi / F);
  const uint32_t s = (uint32_t)(gi % F);
  const uint64_t c = (uint64_t)j * fill + s;
  const bool valid = s < fill && c < n_prev;
  const uint64_t node = (uint64_t)first_this + j;
  t.keys[node * F + s] = valid ? lows_prev[c] : KEY_EMPTY;
  t.vals[node * F + s] = valid ? (uint64_t)(first_prev + c) : 0;
  if (s == 0) {
    const uint64_t c0 = (uint64_t)j * fill;
    NodeMeta m{};
    m.lock = 0;
    m.info = make_info((uint32_t)min<uint64_t>(fill, n_prev - c0), level);
    m.low = lows_prev[c0];
    m.high = (j + 1 < n_this) ? lows_prev[c0 + fill] : KEY_EMPTY;
    m.next = (j + 1 < n_this) ? (uint64_t)(node + 1) : (uint64_t)NODE_NONE;
    t.meta[node] = m;
    lows_out[j] = m.low;
  }
}

// ================================================================== read-only lookup
// G lanes serve one op; lane g of the group holds slots [g*K, g*K+K) of a node.
template <int G>
STM_DEV uint32_t group_sum(uint32_t v) {
#pragma unroll
  for (int off = G / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}

// x[e] for a runtime e, written as a compile-time select tree so the array stays in
// registers (a loop here lets the compiler turn it into an indexed scratch access).
template <int K, int I = 0>
STM_DEV uint64_t select_k(const uint64_t (&x)[K], int e) {
  if constexpr (I == K - 1) {
    return x[I];
  } else {
    return e == I ? x[I] : select_k<K, I + 1>(x, e);
  }
}

// Slot s of the node held by the group (s group-uniform, 0 <= s < F).
template <int F, int G>
STM_DEV uint64_t group_at(const uint64_t (&x)[F / G], int s, int gbase) {
  constexpr int K = F / G;
  return shfl64(select_k<K>(x, s % K), gbase + s / K);
}

template <int F, int G>
STM_DEV int group_count_le(const uint64_t (&x)[F / G], uint64_t key) {
  constexpr int K = F / G;
  uint32_t c = 0;
#pragma unroll
  for (int e = 0; e < K; ++e) c += (x[e] <= key) ? 1u : 0u;
  return (int)group_sum<G>(c);
}

// Slot of key in the leaf held by the group (lane g holds slots g*K .. g*K+K-1, as load_slots
// loads them), -1 if absent.  A leaf's entries are unordered and its free slots hold KEY_EMPTY,
// which is never a key, so one equality test per slot finds it.
template <int F, int G>
STM_DEV int group_find(const uint64_t (&x)[F / G], uint64_t key, int g) {
  constexpr int K = F / G;
  uint32_t hit = 0;  // e + 1 of the slot that holds key in this lane
#pragma unroll
  for (int e = 0; e < K; ++e) hit = x[e] == key ? (uint32_t)(e + 1) : hit;
  return (int)group_sum<G>(hit ? (uint32_t)(g * K) + hit : 0u) - 1;
}

template <int F, int G>
STM_DEV void load_slots(const uint64_t* __restrict__ base, uint32_t node, int g,
                        uint64_t (&x)[F / G]) {
  constexpr int K = F / G;
  const uint64_t* p = base + (size_t)node * F + (size_t)g * K;
#pragma unroll
  for (int e = 0; e < K; ++e) x[e] = p[e];
}

template <int G>
STM_DEV float group_sumf(float v) {
#pragma unroll
  for (int off = G / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, WAVE);
  return v;
}

// Per lane-group state of the learned path: a window of G consecutive directory entries,
// entry base + g in lane g (fence, leaf id, split flag).  Keys arrive sorted, so most keys
// route inside the window with no memory access; the window is refilled from the next
// entries when a key passes its end, and from the model's prediction otherwise.
struct RouteCursor {
  bool valid = false;
  uint32_t base = 0;
  uint64_t f = KEY_EMPTY;  // fence of entry base + g (KEY_EMPTY past the last entry)
  uint32_t lid = NODE_NONE;
  uint32_t pflags = DIR_SPLIT | DIR_PAR_NONE;
};

template <int G>
STM_DEV void window_load(const RouteView& rv, uint32_t base, int g, RouteCursor& c) {
  const uint64_t idx = (uint64_t)base + (uint32_t)g;
  c.valid = true;
  c.base = base;
  c.f = KEY_EMPTY;
  c.lid = NODE_NONE;
  c.pflags = DIR_SPLIT | DIR_PAR_NONE;
  if (idx < rv.L) {
    const DirEntry e = rv.dir[idx];
    c.f = e.fence;
    c.lid = e.lid;
    c.pflags = e.pflags;
  }
}

// Entry of `key` inside the window: true when some entry base + j holds it with its
// successor's fence also in the window (j <= G - 2).
template <int G>
STM_DEV bool window_find(const RouteCursor& c, uint64_t key, int gbase, uint32_t& lid, bool& dirty,
                         uint64_t& hi, uint32_t& cnt_out, uint32_t& par) {
  const uint32_t cnt = group_sum<G>(c.valid && c.f <= key ? 1u : 0u);
  cnt_out = cnt;
  const uint32_t j = cnt > 0 ? cnt - 1 : 0;
  lid = (uint32_t)__shfl((int)c.lid, gbase + (int)j, WAVE);
  const uint32_t pf = (uint32_t)__shfl((int)c.pflags, gbase + (int)j, WAVE);
  dirty = (pf & DIR_SPLIT) != 0;
  par = (pf & DIR_PAR_NONE) == DIR_PAR_NONE ? NODE_NONE : (pf & DIR_PAR_NONE);
  hi = shfl64(c.f, gbase + (int)min(cnt, (uint32_t)G - 1));
  return c.valid && cnt >= 1 && cnt <= (uint32_t)G - 1;
}

// Learned routing of `key` to a directory entry on a tree nobody writes.  Returns true with
// the entry's leaf id, split flag and upper fence; false sends the caller to a root-to-leaf
// descent.  model: 0 = routed without the model, 1 = the model's +/-2 window held the key,
// 2 = the model missed.
template <int F, int G, bool INDEX>
STM_DEV bool learned_route(const RouteView& rv, uint64_t key, int g, int gbase, RouteCursor& c,
                           uint32_t& lid, bool& dirty, uint64_t& hi, int& model, uint32_t& par) {
  model = 0;
  if (rv.L == 0) return false;
  uint32_t cnt = 0;
  if (window_find<G>(c, key, gbase, lid, dirty, hi, cnt, par)) return true;
  if (c.valid && cnt == (uint32_t)G && c.base + G - 1 < rv.L) {
    // Past the window: the next entries (one coalesced load) usually hold the key.
    window_load<G>(rv, c.base + G - 1, g, c);
    if (window_find<G>(c, key, gbase, lid, dirty, hi, cnt, par)) return true;
  }
  if constexpr (INDEX) {
    // Static index: a G-ary search of the directory for the last fence <= key.  The rank lies
    // in [lo, top); each step every lane of the group probes one fence, and the range shrinks
    // to one probe interval.  A range of at most G - 1 entries fits a window with the
    // successor of its last entry.
    uint32_t lo = 0, top = rv.L;
    while (top - lo > (uint32_t)G - 1) {
      const uint32_t step = (top - lo + G - 1) / G;
      const uint32_t q = lo + (uint32_t)g * step;
      const uint32_t below = group_sum<G>(q < top && rv.fences[q] <= key ? 1u : 0u);
      if (below == 0) break;  // the key precedes the first fence: descend instead
      lo += (below - 1) * step;
      top = min(top, lo + step);
    }
    window_load<G>(rv, lo, g, c);
    const bool ok = window_find<G>(c, key, gbase, lid, dirty, hi, cnt, par);
    model = ok ? 1 : 2;
    return ok;
  }
  // The model: root line -> segment -> MLP -> rank p; entries [p-2, p-2+G) are loaded and the
  // key must lie in [p-2, p+2] for a model hit.
  const SegModel* m = rv.segs + root_segment(rv, key);
  const float x = (float)(((double)key - (double)m->klo) * (double)m->inv_w);
  float acc = 0.0f;
  for (int j = g; j < MLP_HIDDEN; j += G)
    acc += m->p[2 * MLP_HIDDEN + j] * fmaxf(m->p[j] * x + m->p[MLP_HIDDEN + j], 0.0f);
  const float y = group_sumf<G>(acc) + m->p[3 * MLP_HIDDEN];
  float rank = (float)m->r0 + y * m->n;
  rank = fminf(fmaxf(rank, 0.0f), (float)(rv.L - 1));  // also maps NaN to 0
  const int64_t p = (int64_t)(rank + 0.5f);
  const uint32_t base = (uint32_t)max<int64_t>(p - ROUTE_WINDOW, 0);
  window_load<G>(rv, base, g, c);
  bool ok = window_find<G>(c, key, gbase, lid, dirty, hi, cnt, par);
  const int64_t r = (int64_t)base + (int64_t)cnt - 1;
  model = (ok && r >= p - ROUTE_WINDOW && r <= p + ROUTE_WINDOW) ? 1 : 2;
  if (!ok) {
    // A miss is usually near: one more window on the side the key lies (before the window:
    // no entry <= key; past it: every entry <= key) before the caller's root-to-leaf descent.
    if (cnt == 0 && base > 0) {
      window_load<G>(rv, base > (uint32_t)G - 1 ? base - (uint32_t)(G - 1) : 0u, g, c);
      ok = window_find<G>(c, key, gbase, lid, dirty, hi, cnt, par);
    } else if (cnt == (uint32_t)G && base + G - 1 < rv.L) {
      window_load<G>(rv, base + G - 1, g, c);
      ok = window_find<G>(c, key, gbase, lid, dirty, hi, cnt, par);
    }
  }
  return ok;
}

// Stripe of the statistics counters a wavefront adds to.
STM_DEV uint32_t wave_stripe() { return blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE; }

// Latency-bound: resident wavefronts hide the node loads.  For F <= 64 and G >= 16 the
// register budget of seven wavefronts per SIMD (72 VGPRs) is requested; the learned variant
// otherwise lands one register above it and loses a seventh of its wavefronts.  Narrower lane
// groups hold more slots per lane and would spill.
template <int F, int G>
constexpr int lookup_min_waves() { return (F <= 64 && G >= 16) ? 7 : 1; }

template <int F, int G, bool LEARNED, bool INDEX>
__global__ __launch_bounds__(256, (lookup_min_waves<F, G>())) void k_lookup(TreeView t, const uint64_t* __restrict__ ukey,
                                                const uint8_t* __restrict__ uop,
                                                const uint32_t* __restrict__ gstart,
                                                const uint32_t* __restrict__ npend,
                                                const uint32_t* __restrict__ sidx,
                                                const BatchCounters* __restrict__ cnt,
                                                uint32_t chunk, uint32_t fill,
                                                uint64_t* __restrict__ out_vals,
                                                uint8_t* __restrict__ out_found,
                                                const RouteHeader* __restrict__ rh,
                                                const uint64_t* __restrict__ fences,
                                                const uint32_t* __restrict__ lids,
                                                const SegModel* __restrict__ segs,
                                                const BatchDesc* __restrict__ desc,
                                                InsHint* __restrict__ ihint,
                                                uint64_t* __restrict__ gval,
                                                uint64_t* __restrict__ fanout,
                                                uint64_t fanout_cap,
                                                SplitState* __restrict__ split,
                                                const StreamAcc* __restrict__ acc) {
  constexpr int K = F / G;
  const bool skip = acc && stream_failed(acc, t.hdr);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    SplitState z{};
    z.refused = NODE_NONE;
    *split = z;
    if (acc) {
      // Every workgroup sees the earlier failure itself; the later kernels see no groups.
      BatchCounters* c = const_cast<BatchCounters*>(cnt);
      c->skipped = skip ? 1u : 0u;
      if (skip) {
        c->n_unique = 0;
        c->n_upserts = 0;
        c->n_fanout = 0;
        c->n_deferred = 0;
      }
    }
  }
  const int lane = lane_id();
  const int g = lane & (G - 1);
  const int gbase = lane - g;
  const uint64_t grp0 = (blockIdx.x * (uint64_t)blockDim.x + threadIdx.x) / G;
  const uint64_t ngroups = (uint64_t)gridDim.x * blockDim.x / G;
  const uint32_t U = skip ? 0u : cnt->n_unique;
  // Every lane group walks one contiguous span of sorted groups, so its cached leaf, parent and
  // directory cursor carry over for the whole span: at least `chunk` of them once there are
  // enough to give every lane group the device holds at once (`fill`) a chunk, fewer below that.
  const uint64_t least = min(chunk, (U + fill - 1) / fill);
  const uint64_t span = max<uint64_t>(max<uint64_t>(least, 1u), (U + ngroups - 1) / ngroups);
  // Groups past the end skip the walk but stay for the wave's statistics reduction.
  const bool active = grp0 * span < U;
  if (desc) {
    out_vals = desc->out_vals;
    out_found = desc->out_found;
  }
  const uint32_t cap = t.capacity;
  const uint32_t root = (uint32_t)min<uint64_t>(t.hdr->root, cap - 1);
  const uint32_t height = (uint32_t)min<uint64_t>(t.hdr->height, 64);

  uint32_t leaf = NODE_NONE;
  uint64_t leaf_hi = 0;
  uint64_t lk[K];
  uint32_t par = NODE_NONE;
  uint64_t par_hi = 0;
  uint64_t pk[K], pv[K];
  RouteView rv{};
  RouteCursor cur;
  uint64_t cur_hi = 0;  // upper fence of the current directory entry
  uint32_t hits = 0, misses = 0;
  uint32_t reads = 0;  // tree nodes this lane group loaded
  if constexpr (LEARNED) rv = route_view(rh, fences, lids, segs, t.dir);

  if (active) {
  const uint32_t i0 = (uint32_t)(grp0 * span);
  const uint32_t i1 = (uint32_t)min<uint64_t>((uint64_t)i0 + span, U);
  for (uint32_t base = i0; base < i1; base += G) {
    // Lane g owns op base + g: its metadata comes in one coalesced round trip, and the
    // sorted position of its first waiting op in a second one that overlaps the walk.
    const uint32_t j = base + g;
    const bool valid = j < i1;
    // Loads from an index clamped into the span (i1 > base), selected afterwards: unconditional
    // loads issue together instead of one guarded round trip after another.
    const uint32_t jc = valid ? j : i1 - 1;
    const uint8_t op_raw = uop[jc];
    const uint64_t key_raw = ukey[jc];
    const uint32_t gs_raw = gstart[jc];
    const uint32_t np_raw = npend[jc];
    __builtin_amdgcn_sched_barrier(0);  // keep all four loads ahead of their first use
    const uint8_t op_l = valid ? op_raw : UOP_SKIP;
    const uint64_t key_l = valid ? key_raw : 0;
    const uint32_t gs_l = valid ? gs_raw : 0;
    const uint32_t np_l = valid ? np_raw : 0;
    const bool mine = op_l == OP_GET;
    // Merged INSERTs are routed too: their leaf is the upsert kernel's starting hint.
    const bool walk = mine || (ihint && op_l == OP_INSERT);
    const uint32_t sx_raw = sidx[gs_l];  // gs_l is a sorted position of the batch
    const uint32_t pos_l = (mine && np_l) ? pos_of(sx_raw) : 0;
    uint64_t vidx_l = 0;  // value slot of op base + g
    uint32_t leaf_l = NODE_NONE, par_l = NODE_NONE;
    bool found_l = false;
    const uint32_t n_sub = min(i1 - base, (uint32_t)G);
    for (uint32_t jj = 0; jj < n_sub; ++jj) {
      if (__shfl((int)walk, gbase + (int)jj, WAVE) == 0) continue;
      const uint64_t key = shfl64(key_l, gbase + (int)jj);
      if (leaf == NODE_NONE || key >= leaf_hi) {
        bool routed = false;
        if constexpr (LEARNED) {
          uint32_t lid = leaf;
          bool dirty = true;
          int model = 0;
          uint32_t rpar = par;
          // Still inside the current directory entry: the leaf split, walk right from it.
          const bool same_entry = leaf != NODE_NONE && key < cur_hi;
          uint64_t hi = cur_hi;
          routed = same_entry ||
                   learned_route<F, G, INDEX>(rv, key, g, gbase, cur, lid, dirty, hi, model, rpar);
          if (routed) {
            par = rpar;  // the level-1 hint recorded for merged INSERTs
            cur_hi = hi;
            leaf = min(lid, cap - 1);
            uint64_t mh = KEY_EMPTY;
            if (dirty) mh = t.meta[leaf].high;
            load_slots<F, G>(t.keys, leaf, g, lk);
            reads += 1;
            if (dirty && key >= mh) {  // the key lives in a right sibling made by a split
              routed = false;
              uint32_t steps = 0;
              for (int step = 0; step < 64; ++step) {
                leaf = (uint32_t)min<uint64_t>(t.meta[leaf].next, cap - 1);
                mh = t.meta[leaf].high;
                steps = (uint32_t)step + 1;
                if (key < mh) {
                  routed = true;
                  break;
                }
              }
              // Rare (only after splits): counted where it happens, so no register carries it.
              if (g == 0) stat_add(t.stats, ST_LEAF_STEPS, blockIdx.x, steps);
              if (routed) {
                load_slots<F, G>(t.keys, leaf, g, lk);
                reads += 1;
              }
              else cur_hi = 0;
            }
            leaf_hi = min(cur_hi, mh);
          } else {
            cur_hi = 0;
          }
          hits += model == 1 ? 1 : 0;
          misses += model == 2 ? 1 : 0;
        }
        if (!routed) {
          if (height <= 1) {
            leaf = root;
            leaf_hi = KEY_EMPTY;
          } else {
            // The learned variant keeps no cached parent: its misses are rare and the
            // registers buy occupancy.
            if (LEARNED || par == NODE_NONE || key >= par_hi) {
              uint32_t node = root;
              uint64_t hi = KEY_EMPTY;
              for (uint32_t lvl = height - 1; lvl > 1; --lvl) {
                uint64_t nk[K], nv[K];
                load_slots<F, G>(t.keys, node, g, nk);
                load_slots<F, G>(t.vals, node, g, nv);
                reads += 1;
                const int s = max(group_count_le<F, G>(nk, key) - 1, 0);
                const uint64_t child = group_at<F, G>(nv, s, gbase);
                const uint64_t nx = (s + 1 < F) ? group_at<F, G>(nk, s + 1, gbase) : KEY_EMPTY;
                hi = min(hi, nx);
                node = (uint32_t)min<uint64_t>(child, cap - 1);
              }
              load_slots<F, G>(t.keys, node, g, pk);
              load_slots<F, G>(t.vals, node, g, pv);
              reads += 1;
              par = node;
              par_hi = hi;
            }
            const int s = max(group_count_le<F, G>(pk, key) - 1, 0);
            leaf = (uint32_t)min<uint64_t>(group_at<F, G>(pv, s, gbase), cap - 1);
            const uint64_t nx = (s + 1 < F) ? group_at<F, G>(pk, s + 1, gbase) : KEY_EMPTY;
            leaf_hi = min(par_hi, nx);
          }
          load_slots<F, G>(t.keys, leaf, g, lk);
          reads += 1;
        }
      }
      const int s = group_find<F, G>(lk, key, g);
      if (g == (int)jj) {
        found_l = s >= 0;
        // The key's slot when found (a new key is appended at the leaf's count).
        vidx_l = (uint64_t)leaf * F + (uint32_t)(found_l ? s : 0);
        leaf_l = leaf;
        par_l = par;
      }
    }
    // The sub-chunk's tail loads go out together, before any of its stores (the vector memory
    // counter counts stores too, so a load issued after a store also waits for the store):
    // the entry count of an INSERT group's leaf, the value a GET group returns.
    const bool hint = walk && !mine;
    uint64_t info = 0;
    if (hint && leaf_l < t.capacity) info = t.meta[leaf_l].info;
    const uint64_t val = (mine && found_l) ? t.vals[vidx_l] : 0;
    if (hint) {
      // The record for the upsert kernels: the op's answer range and leaf, the leaf's entry count
      // now (no writer runs during this kernel), the key's slot in it and the level-1 node last
      // used for routing.
      // field by field, so that the fields need not be live together (registers)
      InsHint* h = ihint + j;
      h->leaf = leaf_l;
      h->pos = (uint32_t)(vidx_l - (uint64_t)leaf_l * F) | (found_l ? UPOS_FOUND : 0u) |
               (min(meta_count(info), 255u) << UPOS_COUNT_SHIFT);
      h->par = par_l;
      h->gs = gs_l;
      h->np = np_l;
    }
    // The answers.  out_found holds 1s already (the front half writes them in input order, whole
    // lines at a time), so only an absent key's op is written here: a byte scattered to its input
    // position is a memory request of its own, as its value is.  With every byte scattered (2^26
    // keys, 2^22 ops at 95/5): this kernel 356 µs instead of 342, k_fold_apply 46.8 instead of 41.7,
    // k_upsert_runs 39.2 instead of 35.7.
    if (mine) {
      if (np_l > FANOUT_DIRECT) {
        // A hot key: its waiting ops are answered by the whole grid (fanout_answers), in
        // chunks queued here, instead of one store after another from this lane.
        gval[j] = val;
        const uint32_t nch = (np_l + FANOUT_CHUNK - 1) / FANOUT_CHUNK;
        const uint32_t c0 = atomicAdd(&const_cast<BatchCounters*>(cnt)->n_fanout, nch);
        for (uint32_t c = 0; c < nch; ++c)
          if ((uint64_t)c0 + c < fanout_cap)
            fanout[c0 + c] = (uint64_t)j | ((uint64_t)(c * FANOUT_CHUNK) << 32) |
                             (found_l ? (1ull << 63) : 0ull);
      } else {
        if (np_l) {
          out_vals[pos_l] = val;
          if (!found_l) out_found[pos_l] = 0;
        }
        for (uint32_t p = 1; p < np_l; ++p) {
          const uint32_t pos = pos_of(sidx[gs_l + p]);
          out_vals[pos] = val;
          if (!found_l) out_found[pos] = 0;
        }
      }
    }
  }
  }  // span
  // One atomic per wavefront and counter: the group leaders' counts summed by readlane.
  uint32_t h = 0, m = 0, nr = 0;
#pragma unroll
  for (int q = 0; q < WAVE; q += G) {
    if constexpr (LEARNED) {
      h += (uint32_t)__builtin_amdgcn_readlane((int)hits, q);
      m += (uint32_t)__builtin_amdgcn_readlane((int)misses, q);
    }
    nr += (uint32_t)__builtin_amdgcn_readlane((int)reads, q);
  }
  if (lane == 0) {
    if (h) stat_add(t.stats, ST_ROUTE_HITS, wave_stripe(), h);
    if (m) stat_add(t.stats, ST_ROUTE_MISSES, wave_stripe(), m);
    if (nr) stat_add(t.stats, ST_NODE_READS, wave_stripe(), nr);
  }
}

// ================================================================== transactional upsert
// A node held by one wavefront: slot s = j*64 + lane.
template <int F>
struct WNode {
  static constexpr int SPL = (F + WAVE - 1) / WAVE;
  uint64_t k[SPL];
  uint64_t v[SPL];
  uint64_t ver;
  uint64_t low, high;
  uint32_t id, count, level, next;
};

template <int F>
STM_DEV uint64_t wave_at(const uint64_t (&x)[WNode<F>::SPL], uint32_t s) {
  uint64_t r = 0;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j)
    if ((s >> 6) == (uint32_t)j) r = readlane64(x[j], (int)(s & 63));
  return r;
}

// Per-lane gather of slot src (any lane, any j); dflt when src is outside [0, F).
template <int F>
STM_DEV uint64_t wgather(const uint64_t (&x)[WNode<F>::SPL], int src, uint64_t dflt) {
  uint64_t r = dflt;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) {
    const uint64_t tv = shfl64(x[j], src & 63);
    if (src >= 0 && src < F && (src >> 6) == j) r = tv;
  }
  return r;
}

template <int F>
STM_DEV uint32_t wave_count_le(const uint64_t (&x)[WNode<F>::SPL], uint64_t key) {
  uint32_t c = 0;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) c += (uint32_t)__popcll(ballot(x[j] <= key));
  return c;
}

// Slot of key in a leaf held by the wavefront (entries unordered, free slots KEY_EMPTY, which
// is never a key); NODE_NONE if absent.  Wave-uniform.
template <int F>
STM_DEV uint32_t wave_find(const uint64_t (&x)[WNode<F>::SPL], uint64_t key) {
  uint32_t s = NODE_NONE;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) {
    const uint64_t m = ballot(x[j] == key);
    if (m) s = (uint32_t)(j * WAVE) + (uint32_t)__builtin_ctzll(m);
  }
  return s;
}

// Rank of each held key among the leaf's first `count` slots (the number of those keys below
// it): its place in key order.  The keys are distinct, so the ranks of the count entries are a
// permutation of [0, count).  One wave-uniform pass over the entries.
template <int F>
STM_DEV void wave_ranks(const uint64_t (&x)[WNode<F>::SPL], uint32_t count,
                        uint32_t (&r)[WNode<F>::SPL]) {
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) r[j] = 0;
  for (uint32_t i = 0; i < count; ++i) {
    const uint64_t ki = wave_at<F>(x, i);
#pragma unroll
    for (int j = 0; j < WNode<F>::SPL; ++j) r[j] += ki < x[j] ? 1u : 0u;
  }
}

// Number of the leaf's first `count` entries below key (wave-uniform).
template <int F>
STM_DEV uint32_t wave_count_below(const uint64_t (&x)[WNode<F>::SPL], uint32_t count, uint64_t key) {
  uint32_t c = 0;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j)
    c += (uint32_t)__popcll(ballot((uint32_t)(j * WAVE + lane_id()) < count && x[j] < key));
  return c;
}

// Slot of parent p that routes key, checked to point at child; NODE_NONE if it does not.
template <int F>
STM_DEV uint32_t parent_slot(const WNode<F>& p, uint64_t key, uint32_t child) {
  const uint32_t cle = wave_count_le<F>(p.k, key);
  if (cle == 0 || cle > p.count) return NODE_NONE;
  if (wave_at<F>(p.v, cle - 1) != (uint64_t)child) return NODE_NONE;
  return cle - 1;
}

// Optimistic read of a node: version word, then (ordered after it) the content.  The
// content is only trusted after the version is re-validated: by the commit CAS for nodes
// the transaction writes, by fences and levels for the nodes it only passes through.
template <int F>
STM_DEV bool tx_read(const TreeView& t, uint32_t id, WNode<F>& n) {
  if (id >= t.capacity) return false;
  NodeMeta* m = t.meta + id;
  const uint64_t w = uniform64(ld_relaxed(&m->lock));
  if (w & 1) return false;
  wave_order();  // content loads issue only after the version word has been read
  const uint64_t info = uniform64(ld_relaxed(&m->info));
  n.low = uniform64(ld_relaxed(&m->low));
  n.high = uniform64(ld_relaxed(&m->high));
  n.next = (uint32_t)uniform64(ld_relaxed(&m->next));
  const uint64_t* kp = t.keys + (size_t)id * F;
  const uint64_t* vp = t.vals + (size_t)id * F;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) {
    const int s = j * WAVE + lane_id();
    if (s < F) {
      n.k[j] = ld_relaxed(kp + s);
      n.v[j] = ld_relaxed(vp + s);
    } else {
      n.k[j] = KEY_EMPTY;
      n.v[j] = 0;
    }
  }
  n.ver = w;
  n.id = id;
  n.count = meta_count(info);
  n.level = meta_level(info);
  return n.count <= (uint32_t)F;
}

// The metadata words of node id (count | level, fences, right sibling), one lane each.
STM_DEV void tx_write_meta(const TreeView& t, uint32_t id, uint32_t count, uint32_t level,
                           uint64_t low, uint64_t high, uint32_t next) {
  NodeMeta* m = t.meta + id;
  const int l = lane_id();
  if (l == 1) st_relaxed(&m->info, make_info(count, level));
  if (l == 2) st_relaxed(&m->low, low);
  if (l == 3) st_relaxed(&m->high, high);
  if (l == 4) st_relaxed(&m->next, (uint64_t)next);
}

template <int F>
STM_DEV void tx_write_node(const TreeView& t, uint32_t id, const uint64_t (&k)[WNode<F>::SPL],
                           const uint64_t (&v)[WNode<F>::SPL], uint32_t count, uint32_t level,
                           uint64_t low, uint64_t high, uint32_t next) {
  uint64_t* kp = t.keys + (size_t)id * F;
  uint64_t* vp = t.vals + (size_t)id * F;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) {
    const int s = j * WAVE + lane_id();
    if (s < F) {
      st_relaxed(kp + s, k[j]);
      st_relaxed(vp + s, v[j]);
    }
  }
  tx_write_meta(t, id, count, level, low, high, next);
}

// Try-lock of up to three version words (two nodes and optionally the tree header).
// Each word must still hold the version the transaction read.  On any failure the words
// already taken are restored to their old value (nothing was written) and false returns.
STM_DEV bool tx_lock(uint64_t* w0, uint64_t v0, uint64_t* w1, uint64_t v1, uint64_t* w2,
                     uint64_t v2) {
  const int l = lane_id();
  uint64_t* w = l == 0 ? w0 : (l == 1 ? w1 : (l == 2 ? w2 : nullptr));
  const uint64_t v = l == 0 ? v0 : (l == 1 ? v1 : v2);
  bool ok = true;
  if (w) ok = cas_u64(w, v, v | 1ull);
  const uint64_t fail = ballot(!ok);
  if (fail) {
    if (w && ok) st_relaxed(w, v);
    return false;
  }
  wave_order();  // the lock bits are held before any content store issues
  return true;
}

STM_DEV void tx_unlock(uint64_t* w0, uint64_t v0, uint64_t* w1, uint64_t v1, uint64_t* w2,
                       uint64_t v2) {
  wave_order();  // every content store is acknowledged before the new versions
  const int l = lane_id();
  uint64_t* w = l == 0 ? w0 : (l == 1 ? w1 : (l == 2 ? w2 : nullptr));
  const uint64_t v = l == 0 ? v0 : (l == 1 ? v1 : v2);
  if (w) st_relaxed(w, v + 2);  // clears the lock bit and bumps the version
}

// Allocates n fresh node ids; NODE_NONE when the pool is exhausted.
STM_DEV uint32_t tx_alloc(const TreeView& t, uint32_t n) {
  uint64_t base = 0;
  if (lane_id() == 0) base = atomicAdd((unsigned long long*)&t.hdr->n_nodes, (unsigned long long)n);
  base = readlane64(base, 0);
  if (base + n > t.capacity) {
    if (lane_id() == 0) atomicOr((unsigned long long*)&t.hdr->error, (unsigned long long)ERR_POOL_FULL);
    return NODE_NONE;
  }
  return (uint32_t)base;
}

// Marks fresh nodes locked (version 0) before they become reachable.
STM_DEV void tx_claim_new(const TreeView& t, uint32_t a, uint32_t b) {
  const int l = lane_id();
  if (l == 0 && a != NODE_NONE) st_relaxed(&t.meta[a].lock, 1ull);
  if (l == 1 && b != NODE_NONE) st_relaxed(&t.meta[b].lock, 1ull);
  wave_order();
}

enum TxResult { TX_DONE = 0, TX_ABORT = 1, TX_RESTART = 2, TX_FAIL = 3, TX_NEED_PARENT = 4 };

struct TxCounters {
  uint32_t commits = 0, aborts = 0, leaf_splits = 0, inner_splits = 0, root_splits = 0;
  uint32_t new_keys = 0;
  uint32_t node_reads = 0;  // nodes read (inner nodes on the way, the leaf)
  bool split_happened = false;  // set by a committed leaf split (the parent changed)
};

// Inserts separator (sep -> rid) right after slot ps of parent p (which has room).
template <int F>
STM_DEV void parent_with_child(const WNode<F>& p, uint32_t ps, uint64_t sep, uint32_t rid,
                               uint64_t (&nk)[WNode<F>::SPL], uint64_t (&nv)[WNode<F>::SPL]) {
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) {
    const int s = j * WAVE + lane_id();
    const uint64_t pk = wgather<F>(p.k, s - 1, KEY_EMPTY);
    const uint64_t pv = wgather<F>(p.v, s - 1, 0);
    const bool keep = s <= (int)ps;
    const bool mine = s == (int)ps + 1;
    nk[j] = keep ? p.k[j] : (mine ? sep : pk);
    nv[j] = keep ? p.v[j] : (mine ? (uint64_t)rid : pv);
  }
}

// Splits the full inner node n (preemptively, its own transaction).  pn is its parent when
// has_par; otherwise n is the root, a new root is made and the header is written.
template <int F>
STM_DEV TxResult tx_split_inner(const TreeView& t, const WNode<F>& n, const WNode<F>& pn,
                                bool has_par, uint64_t hver, uint64_t key, TxCounters& c) {
  constexpr int SPL = WNode<F>::SPL;
  const uint32_t h = F / 2;
  const uint64_t sep = wave_at<F>(n.k, h);
  uint32_t ps = 0;
  if (has_par) {
    if (pn.count >= (uint32_t)F) return TX_ABORT;  // parent filled up meanwhile
    ps = parent_slot<F>(pn, key, n.id);
    if (ps == NODE_NONE) return TX_ABORT;
  }
  uint64_t* hw = has_par ? nullptr : &t.hdr->lock;
  if (!tx_lock(&t.meta[n.id].lock, n.ver, has_par ? &t.meta[pn.id].lock : nullptr,
               has_par ? pn.ver : 0, hw, hver))
    return TX_ABORT;
  const uint32_t nnew = has_par ? 1u : 2u;
  const uint32_t base = tx_alloc(t, nnew);
  if (base == NODE_NONE) {
    tx_unlock(&t.meta[n.id].lock, n.ver - 2, has_par ? &t.meta[pn.id].lock : nullptr,
              has_par ? pn.ver - 2 : 0, hw, hver - 2);
    return TX_FAIL;
  }
  const uint32_t rid = base;
  const uint32_t qid = has_par ? NODE_NONE : base + 1;
  tx_claim_new(t, rid, qid);
  uint64_t lk[SPL], lv[SPL], rk[SPL], rv[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const int s = j * WAVE + lane_id();
    lk[j] = s < (int)h ? n.k[j] : KEY_EMPTY;
    lv[j] = s < (int)h ? n.v[j] : 0;
    const uint64_t gk = wgather<F>(n.k, s + (int)h, KEY_EMPTY);
    const uint64_t gv = wgather<F>(n.v, s + (int)h, 0);
    const bool r_ok = s < (int)(n.count - h);
    rk[j] = r_ok ? gk : KEY_EMPTY;
    rv[j] = r_ok ? gv : 0;
  }
  tx_write_node<F>(t, rid, rk, rv, n.count - h, n.level, sep, n.high, n.next);
  tx_write_node<F>(t, n.id, lk, lv, h, n.level, n.low, sep, rid);
  if (has_par) {
    uint64_t pk[SPL], pv[SPL];
    parent_with_child<F>(pn, ps, sep, rid, pk, pv);
    tx_write_node<F>(t, pn.id, pk, pv, pn.count + 1, pn.level, pn.low, pn.high,
                     pn.next);
  } else {
    uint64_t qk[SPL], qv[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const int s = j * WAVE + lane_id();
      qk[j] = s == 0 ? n.low : (s == 1 ? sep : KEY_EMPTY);
      qv[j] = s == 0 ? (uint64_t)n.id : (s == 1 ? (uint64_t)rid : 0);
    }
    tx_write_node<F>(t, qid, qk, qv, 2, n.level + 1, n.low, n.high, NODE_NONE);
    if (lane_id() == 0) {
      st_relaxed(&t.hdr->root, (uint64_t)qid);
      st_relaxed(&t.hdr->height, (uint64_t)(n.level + 2));
    }
  }
  tx_unlock(&t.meta[n.id].lock, n.ver, has_par ? &t.meta[pn.id].lock : &t.meta[rid].lock,
            has_par ? pn.ver : 0ull, has_par ? &t.meta[rid].lock : &t.hdr->lock, has_par ? 0ull : hver);
  if (!has_par) {
    if (lane_id() == 0) st_relaxed(&t.meta[qid].lock, 2ull);
    c.root_splits++;
  }
  c.inner_splits++;
  c.commits++;
  return TX_RESTART;
}

// Test-and-set lock of a leaf, then its content.  A 64-bit fetch_or takes the lock bit
// without knowing the version; the word it returns is the unlocked version.  Holding the
// lock, the content cannot change, so no re-validation is needed.  On success the caller
// owns the lock and must release it (leaf_release) or commit (version + 2).
template <int F>
STM_DEV bool tx_lock_leaf(const TreeView& t, uint32_t id, WNode<F>& n) {
  if (id >= t.capacity) return false;
  NodeMeta* m = t.meta + id;
  uint64_t old = 0;
  if (lane_id() == 0)
    old = __hip_atomic_fetch_or(&m->lock, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  old = readlane64(old, 0);
  if (old & 1) return false;  // held by another transaction; the word is unchanged
  wave_order();               // content loads issue only after the lock is held
  const uint64_t info = uniform64(ld_relaxed(&m->info));
  n.low = uniform64(ld_relaxed(&m->low));
  n.high = uniform64(ld_relaxed(&m->high));
  n.next = (uint32_t)uniform64(ld_relaxed(&m->next));
  const uint64_t* kp = t.keys + (size_t)id * F;
  const uint64_t* vp = t.vals + (size_t)id * F;
#pragma unroll
  for (int j = 0; j < WNode<F>::SPL; ++j) {
    const int s = j * WAVE + lane_id();
    n.k[j] = s < F ? ld_relaxed(kp + s) : KEY_EMPTY;
    n.v[j] = s < F ? ld_relaxed(vp + s) : 0;
  }
  n.ver = old;
  n.id = id;
  n.count = meta_count(info);
  n.level = meta_level(info);
  return true;
}

// Gives a leaf lock back untouched (nothing was written under it).
STM_DEV void leaf_release(uint64_t* lw, uint64_t ver) {
  if (lane_id() == 0) st_relaxed(lw, ver);
}

// Upsert of (key, val) into leaf n, which this wavefront has locked (tx_lock_leaf).  pn
// is its parent when has_par (else n is the root).  A leaf's entries are unordered: a found key
// takes its value in place, a new one goes to slot count; a full leaf splits by rank, the lower
// half of the F + 1 entries (in key order) staying, the upper half moving to a new right
// sibling, each written in key order.  Every return other than TX_DONE and TX_NEED_PARENT has
// released the leaf; TX_NEED_PARENT keeps it locked.
template <int F>
STM_DEV TxResult tx_leaf_upsert(const TreeView& t, const WNode<F>& n, const WNode<F>& pn,
                                bool has_par, bool par_fresh, uint64_t hver, uint64_t key,
                                uint64_t val, bool& found, uint64_t& old, TxCounters& c) {
  constexpr int SPL = WNode<F>::SPL;
  const int lane = lane_id();
  const uint32_t s = wave_find<F>(n.k, key);
  found = s != NODE_NONE;
  old = found ? wave_at<F>(n.v, s) : 0;
  uint64_t* lw = &t.meta[n.id].lock;
  uint64_t* kp = t.keys + (size_t)n.id * F;
  uint64_t* vp = t.vals + (size_t)n.id * F;
  if (found) {
    if (lane == 0) st_relaxed(vp + s, val);
    tx_unlock(lw, n.ver, nullptr, 0, nullptr, 0);
    c.commits++;
    return TX_DONE;
  }
  if (n.count < (uint32_t)F) {
    if (lane == 0) {
      st_relaxed(kp + n.count, key);
      st_relaxed(vp + n.count, val);
    }
    if (lane == 1) st_relaxed(&t.meta[n.id].info, make_info(n.count + 1, 0));
    tx_unlock(lw, n.ver, nullptr, 0, nullptr, 0);
    c.commits++;
    c.new_keys++;
    return TX_DONE;
  }
  // Full leaf: split F+1 entries into h (left) and F+1-h (right).
  if (has_par && !par_fresh) return TX_NEED_PARENT;
  const uint32_t h = (F + 1) / 2;
  uint32_t ps = 0;
  if (has_par) {
    if (pn.count >= (uint32_t)F) {
      leaf_release(lw, n.ver);
      return TX_ABORT;
    }
    ps = parent_slot<F>(pn, key, n.id);
    if (ps == NODE_NONE) {
      leaf_release(lw, n.ver);
      return TX_ABORT;
    }
  }
  // Places in key order: an old entry's rank among the old ones, plus one above the new key;
  // the new key's place is the number of old entries below it.
  uint32_t r[SPL];
  wave_ranks<F>(n.k, F, r);
#pragma unroll
  for (int j = 0; j < SPL; ++j) r[j] += key < n.k[j] ? 1u : 0u;
  const uint32_t rn = wave_count_below<F>(n.k, F, key);
  // the separator: the entry of place h
  uint64_t cand = 0;
  bool has = false;
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    if (j * WAVE + lane < F && r[j] == h) {
      cand = n.k[j];
      has = true;
    }
  }
  const uint64_t sep = rn == h ? key : readlane64(cand, __builtin_ctzll(ballot(has) | (1ull << 63)));
  uint64_t* pw = has_par ? &t.meta[pn.id].lock : nullptr;
  uint64_t* hw = has_par ? nullptr : &t.hdr->lock;
  if (!tx_lock(pw, has_par ? pn.ver : 0, hw, hver, nullptr, 0)) {
    leaf_release(lw, n.ver);
    return TX_ABORT;
  }
  const uint32_t base = tx_alloc(t, has_par ? 1u : 2u);
  if (base == NODE_NONE) {
    tx_unlock(lw, n.ver - 2, pw, has_par ? pn.ver - 2 : 0, hw, hver - 2);
    return TX_FAIL;
  }
  const uint32_t rid = base;
  const uint32_t qid = has_par ? NODE_NONE : base + 1;
  tx_claim_new(t, rid, qid);
  uint64_t* rkp = t.keys + (size_t)rid * F;
  uint64_t* rvp = t.vals + (size_t)rid * F;
  // Every entry to its place: [0, h) in this leaf, [h, F+1) in the right sibling.  The left
  // leaf's slots from h up are freed; the right sibling's slots past its F+1-h entries are free.
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const uint32_t sl = (uint32_t)(j * WAVE + lane);
    if (sl < (uint32_t)F) {
      const uint32_t to = r[j];
      if (to >= h) {
        st_relaxed(rkp + (to - h), n.k[j]);
        st_relaxed(rvp + (to - h), n.v[j]);
      } else if (to != sl) {
        st_relaxed(kp + to, n.k[j]);
        st_relaxed(vp + to, n.v[j]);
      }
      if (sl >= h) st_relaxed(kp + sl, KEY_EMPTY);
      if (sl >= F + 1 - h) st_relaxed(rkp + sl, KEY_EMPTY);
    }
  }
  if (lane == 0) {
    if (rn >= h) {
      st_relaxed(rkp + (rn - h), key);
      st_relaxed(rvp + (rn - h), val);
    } else {
      st_relaxed(kp + rn, key);
      st_relaxed(vp + rn, val);
    }
  }
  tx_write_meta(t, rid, F + 1 - h, 0, sep, n.high, n.next);
  tx_write_meta(t, n.id, h, 0, n.low, sep, rid);
  if (has_par) {
    uint64_t pk[SPL], pv[SPL];
    parent_with_child<F>(pn, ps, sep, rid, pk, pv);
    tx_write_node<F>(t, pn.id, pk, pv, pn.count + 1, pn.level, pn.low, pn.high,
                     pn.next);
    tx_unlock(lw, n.ver, pw, pn.ver, &t.meta[rid].lock, 0ull);
  } else {
    uint64_t qk[SPL], qv[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const int q = j * WAVE + lane;
      qk[j] = q == 0 ? n.low : (q == 1 ? sep : KEY_EMPTY);
      qv[j] = q == 0 ? (uint64_t)n.id : (q == 1 ? (uint64_t)rid : 0);
    }
    tx_write_node<F>(t, qid, qk, qv, 2, 1, n.low, n.high, NODE_NONE);
    if (lane == 0) {
      st_relaxed(&t.hdr->root, (uint64_t)qid);
      st_relaxed(&t.hdr->height, 2ull);
    }
    tx_unlock(lw, n.ver, &t.meta[rid].lock, 0ull, &t.hdr->lock, hver);
    if (lane == 0) st_relaxed(&t.meta[qid].lock, 2ull);
    c.root_splits++;
  }
  if (t.rank_of && lane == 0) {
    const uint32_t rr = t.rank_of[n.id];
    if (rr != NODE_NONE) t.dir[rr].pflags |= DIR_SPLIT;
  }
  c.leaf_splits++;
  c.commits++;
  c.new_keys++;
  c.split_happened = true;
  return TX_DONE;
}

// The inner node of level 1 that routed the wavefront's previous upsert.  Its content may
// be stale by the time it is used again; a stale route is caught by the leaf's fence check
// (and, for a split, by re-reading the parent with its version).
template <int F>
struct ParentCache {
  WNode<F> n;
  bool valid = false;
  bool fresh = false;  // read (version, then content) during the current attempt
};

// Routing part of an upsert attempt: the leaf that holds key, locked (tx_lock_leaf) into cur,
// with its parent par when has_par (read with its version during this attempt when
// par_fresh) and, after a descent from the root, the header version hver.  TX_DONE: the
// leaf is locked and its fences hold key.  Any other result holds no lock.
template <int F>
STM_DEV TxResult tx_route_leaf(const TreeView& t, uint64_t key, TxCounters& c, ParentCache<F>& pc,
                               uint32_t par_hint, WNode<F>& par, WNode<F>& cur, bool& has_par,
                               bool& par_fresh, uint64_t& hver) {
  has_par = false;
  par_fresh = false;
  hver = 0;
  uint32_t leaf_id;
  pc.fresh = false;
  if (!(pc.valid && key >= pc.n.low && key < pc.n.high) && par_hint < t.capacity) {
    // The level-1 node the lookup kernel routed this key through: one read instead of a
    // descent from the root.  Its fences and level check it; the leaf's fences check the route.
    pc.valid = tx_read<F>(t, par_hint, pc.n) && pc.n.level == 1 && key >= pc.n.low && key < pc.n.high;
    pc.fresh = pc.valid;
    c.node_reads++;
  }
  if (pc.valid && key >= pc.n.low && key < pc.n.high) {
    // Route through the cached level-1 node; the tree never loses a level, so no header
    // read is needed.  The leaf's fences validate the route.
    const uint32_t cle = wave_count_le<F>(pc.n.k, key);
    if (cle == 0 || cle > pc.n.count) {
      pc.valid = false;
      return TX_ABORT;
    }
    leaf_id = (uint32_t)wave_at<F>(pc.n.v, cle - 1);
    par = pc.n;
    has_par = true;
    par_fresh = pc.fresh;
  } else {
    hver = uniform64(ld_relaxed(&t.hdr->lock));
    if (hver & 1) return TX_ABORT;
    wave_order();
    const uint32_t root = (uint32_t)uniform64(ld_relaxed(&t.hdr->root));
    const uint32_t height = (uint32_t)uniform64(ld_relaxed(&t.hdr->height));
    if (height == 0 || height > 64) return TX_ABORT;
    leaf_id = root;
    if (height >= 2) {
      uint32_t id = root;
      for (uint32_t lvl = height - 1; lvl >= 1; --lvl) {
        c.node_reads++;
        if (!tx_read<F>(t, id, cur)) return TX_ABORT;
        if (cur.level != lvl || key < cur.low || key >= cur.high) return TX_ABORT;
        if (cur.count >= (uint32_t)F) {
          pc.valid = false;
          return tx_split_inner<F>(t, cur, par, has_par, hver, key, c);
        }
        const uint32_t cle = wave_count_le<F>(cur.k, key);
        if (cle == 0 || cle > cur.count) return TX_ABORT;
        const uint64_t child = wave_at<F>(cur.v, cle - 1);
        if (child >= t.capacity) return TX_ABORT;
        par = cur;
        has_par = true;
        id = (uint32_t)child;
      }
      pc.n = par;
      pc.valid = true;
      par_fresh = true;
      leaf_id = id;
    }
  }
  c.node_reads++;
  if (!tx_lock_leaf<F>(t, leaf_id, cur)) return TX_ABORT;
  if (cur.level != 0 || cur.count > (uint32_t)F || key < cur.low || key >= cur.high) {
    leaf_release(&t.meta[leaf_id].lock, cur.ver);
    pc.valid = false;
    return TX_ABORT;
  }
  return TX_DONE;
}

// Re-reads the parent of the locked leaf cur with its version before a split (the leaf stays
// locked); false releases the leaf.
template <int F>
STM_DEV bool tx_fresh_parent(const TreeView& t, uint64_t key, const WNode<F>& cur, WNode<F>& par,
                             TxCounters& c, ParentCache<F>& pc) {
  c.node_reads++;
  if (!tx_read<F>(t, par.id, par) || par.level != 1 || key < par.low || key >= par.high) {
    leaf_release(&t.meta[cur.id].lock, cur.ver);
    pc.valid = false;
    return false;
  }
  return true;
}

// One attempt of the upsert transaction for (key, val).
template <int F>
STM_DEV TxResult tx_upsert_attempt(const TreeView& t, uint64_t key, uint64_t val, bool& found,
                                   uint64_t& old, TxCounters& c, ParentCache<F>& pc,
                                   uint32_t par_hint) {
  WNode<F> par, cur;
  bool has_par, par_fresh;
  uint64_t hver;
  TxResult r = tx_route_leaf<F>(t, key, c, pc, par_hint, par, cur, has_par, par_fresh, hver);
  if (r != TX_DONE) return r;
  r = tx_leaf_upsert<F>(t, cur, par, has_par, par_fresh, hver, key, val, found, old, c);
  if (r == TX_NEED_PARENT) {
    // The leaf splits: the parent's current version and content are needed.
    if (!tx_fresh_parent<F>(t, key, cur, par, c, pc)) return TX_ABORT;
    r = tx_leaf_upsert<F>(t, cur, par, true, true, hver, key, val, found, old, c);
  }
  if (r != TX_DONE || c.split_happened) pc.valid = false;
  c.split_happened = false;
  return r;
}

// Merged upsert of the ops of lanes R into leaf n, which this wavefront has locked (each lane's
// key k_l and value v_l; keys are distinct): one transaction writes them all.  A leaf's entries
// are unordered: each op's key is looked up by equality over the leaf's slots, a key already
// present takes its new value in place, and the new keys are appended from slot count in lane
// order.  With T = count + new keys <= F the leaf is rewritten in place; with F < T <= 2F it
// splits by rank, the lower T/2 entries (in key order) staying, the rest moving to a new right
// sibling, each half written in key order, and one separator goes into the parent, as the
// single-op split does.  Returns as tx_leaf_upsert; found_l / old_l are each lane's answer.
template <int F>
STM_DEV TxResult tx_leaf_merge(const TreeView& t, const WNode<F>& n, const WNode<F>& pn,
                               bool has_par, bool par_fresh, uint64_t hver, uint64_t key0,
                               uint64_t R, uint64_t k_l, uint64_t v_l, bool& found_l,
                               uint64_t& old_l, TxCounters& c) {
  constexpr int SPL = WNode<F>::SPL;
  const int lane = lane_id();
  const bool mine = (R >> lane) & 1ull;
  uint64_t* lw = &t.meta[n.id].lock;
  // The ops' keys in the leaf, one op at a time (wave-uniform): uv = the values after the found
  // ops' updates, fmask = the found ops, each found lane's old value.
  uint64_t uv[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) uv[j] = n.v[j];
  uint64_t fmask = 0;
  uint64_t oldv = 0;
  for (uint64_t rest = R; rest; rest &= rest - 1) {
    const int i = __builtin_ctzll(rest);
    const uint64_t ki = readlane64(k_l, i);
    const uint32_t s = wave_find<F>(n.k, ki);
    if (s != NODE_NONE) {
      const uint64_t vi = readlane64(v_l, i);
      const uint64_t ov = wave_at<F>(n.v, s);
#pragma unroll
      for (int j = 0; j < SPL; ++j)
        if ((uint32_t)(j * WAVE + lane) == s) uv[j] = vi;
      fmask |= 1ull << i;
      if (lane == i) oldv = ov;
    }
  }
  const bool fnd = (fmask >> lane) & 1ull;
  const uint64_t newm = R & ~fmask;
  const uint32_t ins = (uint32_t)__popcll(newm);
  const uint32_t T = n.count + ins;
  found_l = fnd;
  old_l = fnd ? oldv : 0;
  uint64_t* kp = t.keys + (size_t)n.id * F;
  uint64_t* vp = t.vals + (size_t)n.id * F;
  if (T <= (uint32_t)F) {
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const uint32_t sl = (uint32_t)(j * WAVE + lane);
      if (sl < n.count && uv[j] != n.v[j]) st_relaxed(vp + sl, uv[j]);
    }
    if (mine && !fnd) {
      const uint32_t P = n.count + (uint32_t)__popcll(newm & lanemask_lt());
      st_relaxed(kp + P, k_l);
      st_relaxed(vp + P, v_l);
    }
    if (ins && lane == 1) st_relaxed(&t.meta[n.id].info, make_info(T, 0));
    tx_unlock(lw, n.ver, nullptr, 0, nullptr, 0);
    c.commits++;
    c.new_keys += ins;
    return TX_DONE;
  }
  // Split: entries at places [0, h) in key order stay, [h, T) move to a new right sibling.
  if (has_par && !par_fresh) return TX_NEED_PARENT;
  const uint32_t h = T / 2;
  uint32_t ps = 0;
  if (has_par) {
    if (pn.count >= (uint32_t)F) {
      leaf_release(lw, n.ver);
      return TX_ABORT;
    }
    ps = parent_slot<F>(pn, key0, n.id);
    if (ps == NODE_NONE) {
      leaf_release(lw, n.ver);
      return TX_ABORT;
    }
  }
  // Places in key order: for an old entry, the old entries below it plus the new keys below it;
  // for a new key, the same.
  uint32_t r[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) r[j] = 0;
  uint32_t rn = 0;  // per lane: entries below k_l
  for (uint32_t i = 0; i < n.count; ++i) {
    const uint64_t ki = wave_at<F>(n.k, i);
#pragma unroll
    for (int j = 0; j < SPL; ++j) r[j] += ki < n.k[j] ? 1u : 0u;
    rn += ki < k_l ? 1u : 0u;
  }
  for (uint64_t rest = newm; rest; rest &= rest - 1) {
    const uint64_t ki = readlane64(k_l, __builtin_ctzll(rest));
#pragma unroll
    for (int j = 0; j < SPL; ++j) r[j] += ki < n.k[j] ? 1u : 0u;
    rn += ki < k_l ? 1u : 0u;
  }
  // the separator: the entry whose place is h
  uint64_t cand = 0;
  bool has = false;
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const uint32_t sl = (uint32_t)(j * WAVE + lane);
    if (sl < n.count && r[j] == h) {
      cand = n.k[j];
      has = true;
    }
  }
  if (mine && !fnd && rn == h) {
    cand = k_l;
    has = true;
  }
  const uint64_t sep = readlane64(cand, __builtin_ctzll(ballot(has) | (1ull << 63)));
  uint64_t* pw = has_par ? &t.meta[pn.id].lock : nullptr;
  uint64_t* hw = has_par ? nullptr : &t.hdr->lock;
  if (!tx_lock(pw, has_par ? pn.ver : 0, hw, hver, nullptr, 0)) {
    leaf_release(lw, n.ver);
    return TX_ABORT;
  }
  const uint32_t base = tx_alloc(t, has_par ? 1u : 2u);
  if (base == NODE_NONE) {
    tx_unlock(lw, n.ver - 2, pw, has_par ? pn.ver - 2 : 0, hw, hver - 2);
    return TX_FAIL;
  }
  const uint32_t rid = base;
  const uint32_t qid = has_par ? NODE_NONE : base + 1;
  tx_claim_new(t, rid, qid);
  uint64_t* rkp = t.keys + (size_t)rid * F;
  uint64_t* rvp = t.vals + (size_t)rid * F;
  // Every entry to its place; the left leaf's old slots from h up are freed, and the right
  // sibling's slots past its T - h entries are free.
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const uint32_t sl = (uint32_t)(j * WAVE + lane);
    if (sl < n.count) {
      const uint32_t to = r[j];
      if (to >= h) {
        st_relaxed(rkp + (to - h), n.k[j]);
        st_relaxed(rvp + (to - h), uv[j]);
      } else if (to != sl || uv[j] != n.v[j]) {
        st_relaxed(kp + to, n.k[j]);
        st_relaxed(vp + to, uv[j]);
      }
      if (sl >= h) st_relaxed(kp + sl, KEY_EMPTY);  // the left node ends at h
    }
    if (sl >= T - h && sl < (uint32_t)F) st_relaxed(rkp + sl, KEY_EMPTY);
  }
  if (mine && !fnd) {
    if (rn >= h) {
      st_relaxed(rkp + (rn - h), k_l);
      st_relaxed(rvp + (rn - h), v_l);
    } else {
      st_relaxed(kp + rn, k_l);
      st_relaxed(vp + rn, v_l);
    }
  }
  tx_write_meta(t, rid, T - h, 0, sep, n.high, n.next);
  tx_write_meta(t, n.id, h, 0, n.low, sep, rid);
  if (has_par) {
    uint64_t pk[SPL], pv[SPL];
    parent_with_child<F>(pn, ps, sep, rid, pk, pv);
    tx_write_node<F>(t, pn.id, pk, pv, pn.count + 1, pn.level, pn.low, pn.high, pn.next);
    tx_unlock(lw, n.ver, pw, pn.ver, &t.meta[rid].lock, 0ull);
  } else {
    uint64_t qk[SPL], qv[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const int sl = j * WAVE + lane;
      qk[j] = sl == 0 ? n.low : (sl == 1 ? sep : KEY_EMPTY);
      qv[j] = sl == 0 ? (uint64_t)n.id : (sl == 1 ? (uint64_t)rid : 0);
    }
    tx_write_node<F>(t, qid, qk, qv, 2, 1, n.low, n.high, NODE_NONE);
    if (lane == 0) {
      st_relaxed(&t.hdr->root, (uint64_t)qid);
      st_relaxed(&t.hdr->height, 2ull);
    }
    tx_unlock(lw, n.ver, &t.meta[rid].lock, 0ull, &t.hdr->lock, hver);
    if (lane == 0) st_relaxed(&t.meta[qid].lock, 2ull);
    c.root_splits++;
  }
  if (t.rank_of && lane == 0) {
    const uint32_t r = t.rank_of[n.id];
    if (r != NODE_NONE) t.dir[r].pflags |= DIR_SPLIT;
  }
  c.leaf_splits++;
  c.commits++;
  c.new_keys += ins;
  c.split_happened = true;
  return TX_DONE;
}

// One attempt of a merged upsert: routes key0 (the lowest remaining lane's key) to its leaf,
// locks it and merges every remaining op of the round (todo) whose key the leaf's fences
// hold, at most F of them.  On TX_DONE, done is the lanes whose ops committed.  With a leaf
// hint (the leaf the lookup kernel found) and its level-1 hint the leaf is locked directly:
// fast-path commits never split, so the leaf still holds the key unless a transaction of this
// launch split it, which its fences show; a split then reads the hinted parent with its version
// and checks that it points at the leaf.
template <int F>
STM_DEV TxResult tx_merge_attempt(const TreeView& t, uint64_t key0, uint64_t todo, uint64_t k_l,
                                  uint64_t v_l, TxCounters& c, ParentCache<F>& pc,
                                  uint32_t par_hint, uint32_t leaf_hint, uint64_t& done,
                                  bool& found_l, uint64_t& old_l) {
  WNode<F> par, cur;
  bool has_par = false, par_fresh = false, direct = false;
  uint64_t hver = 0;
  TxResult r;
  if (leaf_hint < t.capacity && par_hint < t.capacity) {
    c.node_reads++;
    if (!tx_lock_leaf<F>(t, leaf_hint, cur)) return TX_ABORT;  // locked by another transaction
    if (cur.level == 0 && cur.count <= (uint32_t)F && key0 >= cur.low && key0 < cur.high) {
      direct = true;
      has_par = true;
      par.id = par_hint;
    } else {
      leaf_release(&t.meta[leaf_hint].lock, cur.ver);
    }
  }
  if (!direct) {
    r = tx_route_leaf<F>(t, key0, c, pc, par_hint, par, cur, has_par, par_fresh, hver);
    if (r != TX_DONE) return r;
  }
  uint64_t R = ballot(((todo >> lane_id()) & 1ull) && k_l >= cur.low && k_l < cur.high);
  if constexpr (F < WAVE) {
    // at most F ops, so that T <= 2F (the lowest lanes: key0's lane is the lowest of todo)
    uint64_t keep = 0;
    for (int q = 0; q < F && R; ++q) {
      keep |= R & (~R + 1);
      R &= R - 1;
    }
    R = keep;
  }
  r = tx_leaf_merge<F>(t, cur, par, has_par, par_fresh, hver, key0, R, k_l, v_l, found_l, old_l, c);
  if (r == TX_NEED_PARENT) {
    if (!tx_fresh_parent<F>(t, key0, cur, par, c, pc)) return TX_ABORT;
    r = tx_leaf_merge<F>(t, cur, par, true, true, hver, key0, R, k_l, v_l, found_l, old_l, c);
  }
  if (r != TX_DONE || c.split_happened) pc.valid = false;
  c.split_happened = false;
  done = r == TX_DONE ? R : 0;
  return r;
}

STM_DEV void backoff(uint32_t attempt) {
  const uint32_t spins = min(attempt, 32u);
  for (uint32_t i = 0; i < spins; ++i) __builtin_amdgcn_s_sleep(4);
}

// Runs one merged upsert to completion (or gives up after max_attempts) and answers the
// np ops of its group that wait for the tree (sorted positions gs .. gs+np-1).
template <int F>
STM_DEV bool run_upsert(const TreeView& t, uint64_t key, uint64_t val, uint32_t gs, uint32_t np,
                        const uint32_t* __restrict__ sidx, uint64_t* __restrict__ out_vals,
                        uint8_t* __restrict__ out_found, uint32_t max_attempts, TxCounters& c,
                        ParentCache<F>& pc, uint32_t par_hint = NODE_NONE) {
  bool found = false;
  uint64_t old = 0;
  uint32_t aborts = 0, restarts = 0;
  for (;;) {
    // The hint is only tried on the first attempt; retries descend from the root.
    const TxResult r = tx_upsert_attempt<F>(t, key, val, found, old, c, pc,
                                            aborts + restarts == 0 ? par_hint : NODE_NONE);
    if (r == TX_DONE) break;
    if (r == TX_FAIL) {  // pool exhausted: error bit raised, op dropped, answered as absent
      found = false;
      old = 0;
      break;
    }
    if (r == TX_ABORT) {
      c.aborts++;
      if (++aborts >= max_attempts) return false;
      backoff(aborts);
    } else if (++restarts >= 4 * max_attempts) {  // TX_RESTART after a preemptive split
      return false;
    }
  }
  if (out_vals) {
    for (uint32_t p = lane_id(); p < np; p += WAVE) {
      const uint32_t pos = pos_of(sidx[gs + p]);
      out_vals[pos] = old;
      out_found[pos] = found ? 1 : 0;
    }
  }
  return true;
}


STM_DEV void flush_counters(const TreeView& t, const TxCounters& c) {
  if (lane_id() == 0) {
    const uint32_t w = wave_stripe();
    stat_add(t.stats, ST_COMMITS, w, c.commits);
    stat_add(t.stats, ST_ABORTS, w, c.aborts);
    stat_add(t.stats, ST_LEAF_SPLITS, w, c.leaf_splits);
    stat_add(t.stats, ST_INNER_SPLITS, w, c.inner_splits);
    stat_add(t.stats, ST_ROOT_SPLITS, w, c.root_splits);
    stat_add(t.stats, ST_KEYS, w, c.new_keys);
    stat_add(t.stats, ST_NODE_READS, w, c.node_reads);
  }
}

// Also adds the wavefront's leaf splits to the batch's counter (the host's retrain trigger).
STM_DEV void flush_counters(const TreeView& t, const TxCounters& c, BatchCounters* cnt) {
  if (lane_id() == 0 && c.leaf_splits) atomicAdd(&cnt->leaf_splits, (uint32_t)c.leaf_splits);
  flush_counters(t, c);
}

// Answers of the hot GET groups the lookup kernel queued (more than FANOUT_DIRECT waiting
// ops): chunk c of the queue is op range [first, first + FANOUT_CHUNK) of group g's waiting
// ops, written by one workgroup, chunks spread over the grid.  Runs at the start of k_upsert_runs,
// whose writes (INSERT groups' answers) never touch a GET group's ops.  Reference:
// the per-op answer write-back, writebackAns (src/gpu-stm-tree-v38/bpt-gpustm-kernel-aux.cuh:46-56).
STM_DEV void fanout_answers(const uint64_t* __restrict__ fanout, uint64_t cap,
                            const BatchCounters* cnt, const uint32_t* __restrict__ gstart,
                            const uint32_t* __restrict__ npend, const uint64_t* __restrict__ gval,
                            const uint32_t* __restrict__ sidx, uint64_t* __restrict__ out_vals,
                            uint8_t* __restrict__ out_found) {
  const uint32_t nc = (uint32_t)min<uint64_t>(cnt->n_fanout, cap);
  for (uint32_t c = blockIdx.x; c < nc; c += gridDim.x) {
    const uint64_t e = fanout[c];
    const uint32_t g = (uint32_t)e;
    const uint32_t first = (uint32_t)(e >> 32) & 0x7fffffffu;
    const bool found = e >> 63;
    const uint32_t gs = gstart[g];
    const uint32_t end = min(npend[g], first + FANOUT_CHUNK);
    const uint64_t v = gval[g];
    for (uint32_t p = first + threadIdx.x; p < end; p += blockDim.x) {
      const uint32_t pos = pos_of(sidx[gs + p]);
      out_vals[pos] = v;
      if (!found) out_found[pos] = 0;
    }
  }
}

// Answers of the committed ops of a round (lanes with ans): a lane writes its own group's few
// waiting ops (np of them from sorted position gs, p0 the first one's input position); a group
// with many (a hot key) is written by the whole wavefront.  Called by every lane of the wavefront.
STM_DEV void write_upsert_answers(bool ans, bool found, uint64_t old, uint32_t gs, uint32_t np,
                                  uint32_t p0, const uint32_t* __restrict__ sidx,
                                  uint64_t* __restrict__ out_vals, uint8_t* __restrict__ out_found) {
  const bool many = ans && np > 8;
  if (ans && !many) {
    for (uint32_t p = 0; p < np; ++p) {
      const uint32_t pos = p == 0 ? p0 : pos_of(sidx[gs + p]);
      out_vals[pos] = old;
      if (!found) out_found[pos] = 0;
    }
  }
  for (uint64_t bm = ballot(many); bm; bm &= bm - 1) {
    const int b = __builtin_ctzll(bm);
    const uint32_t gsb = __builtin_amdgcn_readlane(gs, b);
    const uint32_t npb = __builtin_amdgcn_readlane(np, b);
    const uint64_t ob = readlane64(old, b);
    const bool fb = __builtin_amdgcn_readlane(found ? 1 : 0, b) != 0;
    for (uint32_t p = lane_id(); p < npb; p += WAVE) {
      const uint32_t pos = pos_of(sidx[gsb + p]);
      out_vals[pos] = ob;
      if (!fb) out_found[pos] = 0;
    }
  }
}

// Leaf of insert-list entry e as the lookup kernel routed it.
STM_DEV uint32_t entry_leaf(const uint32_t* __restrict__ ilist, const InsHint* __restrict__ ihint,
                            uint32_t e) {
  return ihint[ilist[e]].leaf;
}

// First entry after `from` whose leaf differs from the leaf of `from` (N if none): entries of a
// leaf are neighbours in the list, and every lane probes one entry of the range per step.
STM_DEV uint32_t run_end(const uint32_t* __restrict__ ilist, const InsHint* __restrict__ ihint,
                         uint32_t from, uint32_t N, uint32_t leaf) {
  const uint32_t lane = (uint32_t)lane_id();
  uint32_t lo = from + 1, hi = N;  // the answer lies in [lo, hi]
  while (hi - lo > (uint32_t)WAVE) {
    const uint32_t step = (hi - lo + WAVE - 1) / WAVE;
    const uint32_t at = lo + lane * step;
    const uint32_t same = (uint32_t)__popcll(
        ballot(at < hi && entry_leaf(ilist, ihint, min(at, N - 1)) == leaf));
    if (same == 0) return lo;
    const uint32_t up = min(hi, lo + same * step);
    lo += (same - 1) * step + 1;
    hi = up;
  }
  const uint32_t at = lo + lane;
  return lo + (uint32_t)__popcll(ballot(at < hi && entry_leaf(ilist, ihint, min(at, N - 1)) == leaf));
}

// The node at `level` (1 or more) whose range holds key, by a descent from the root; NODE_NONE if
// the tree is not that high.  For kernels in which no node above that level is being written.
template <int F>
STM_DEV uint32_t find_at_level(const TreeView& t, uint64_t key, uint32_t level) {
  constexpr int SPL = WNode<F>::SPL;
  uint32_t node = (uint32_t)uniform64(t.hdr->root);
  const uint32_t height = (uint32_t)min<uint64_t>(uniform64(t.hdr->height), 64);
  if (height <= level) return NODE_NONE;
  for (uint32_t lvl = height - 1; lvl > level && node < t.capacity; --lvl) {
    uint64_t k[SPL], v[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
      const int sl = j * WAVE + lane_id();
      const size_t at = (size_t)node * F + (size_t)min(sl, F - 1);
      const uint64_t kk = t.keys[at];
      v[j] = t.vals[at];
      k[j] = sl < F ? kk : KEY_EMPTY;
    }
    const uint32_t cle = wave_count_le<F>(k, key);
    node = (uint32_t)wave_at<F>(v, cle ? cle - 1 : 0);
  }
  return node < t.capacity ? node : NODE_NONE;
}

// How the T entries of an overfull node are spread over nl nodes: node j gets entries [bound(j),
// bound(j + 1)) in key order, one more in the first T mod nl nodes.  Node 0 is the old one, node
// j > 0 has id base + j - 1.
struct Spread {
  uint32_t node, base, nl, per, more;
  STM_DEV Spread(uint32_t T, uint32_t nl_, uint32_t node_, uint32_t base_)
      : node(node_), base(base_), nl(nl_), per(T / nl_), more(T % nl_) {}
  STM_DEV uint32_t bound(uint32_t j) const { return j * per + min(j, more); }
  STM_DEV uint32_t id(uint32_t j) const { return j == 0 ? node : base + j - 1; }
  // Node of the entry of rank r.
  STM_DEV uint32_t part(uint32_t r) const {
    const uint32_t q = more * (per + 1);
    return r < q ? r / (per + 1) : more + (r - q) / per;
  }
};

// Nodes an overfull node of T entries is spread over: three quarters full each, as built.
template <int F>
STM_DEV uint32_t spread_nodes(uint32_t T) {
  constexpr uint32_t PER = F - F / 4;
  return (T + PER - 1) / PER;
}

// One entry to its place; the first entry of a new node is its low fence and the high fence of the
// node before it.
template <int F>
STM_DEV void spread_entry(const TreeView& t, const Spread& sp, uint32_t r, uint64_t k, uint64_t v) {
  const uint32_t j = sp.part(r);
  const uint32_t slot = r - sp.bound(j);
  const size_t at = (size_t)sp.id(j) * F + slot;
  t.keys[at] = k;
  t.vals[at] = v;
  if (slot == 0 && j > 0) {
    st_relaxed(&t.meta[sp.id(j)].low, k);
    st_relaxed(&t.meta[sp.id(j - 1)].high, k);
  }
}

// The rest of a spread, by `waves` wavefronts of which this is the wave-th: free slots, counts,
// sibling links, the last node's high fence, and the note for the parent.  used: entries the old
// node held.
template <int F>
STM_DEV void spread_finish(const TreeView& t, const Spread& sp, uint32_t level, uint32_t used,
                           uint64_t high, uint64_t next, uint32_t wave = 0, uint32_t waves = 1) {
  const uint32_t lane = (uint32_t)lane_id();
  for (uint32_t j = wave; j < sp.nl; j += waves) {
    const uint32_t n = sp.bound(j + 1) - sp.bound(j);
    const uint32_t end = j == 0 ? used : (uint32_t)F;
    for (uint32_t sl = n + lane; sl < end; sl += WAVE) {
      t.keys[(size_t)sp.id(j) * F + sl] = KEY_EMPTY;
      t.vals[(size_t)sp.id(j) * F + sl] = 0;
    }
  }
  for (uint32_t j = wave * WAVE + lane; j < sp.nl; j += waves * WAVE) {
    NodeMeta* m = t.meta + sp.id(j);
    const bool last = j + 1 == sp.nl;
    st_relaxed(&m->info, make_info(sp.bound(j + 1) - sp.bound(j), level));
    st_relaxed(&m->next, last ? next : (uint64_t)sp.id(j + 1));
    if (last) st_relaxed(&m->high, high);
    if (j == 0 && sp.nl > 1) st_relaxed(&m->made, (uint64_t)sp.base | ((uint64_t)(sp.nl - 1) << 32));
  }
}

// Splits the overfull leaf of a run (entries unordered, `newm` the lanes with new keys, in key
// order) over nl nodes.  The leaf belongs to this wavefront; nothing is locked and the parent is
// not touched.
template <int F>
STM_DEV void split_run(const TreeView& t, uint32_t leaf, uint32_t base, uint32_t nl, uint64_t newm,
                       uint64_t key, uint64_t val) {
  constexpr int SPL = WNode<F>::SPL;
  const uint32_t lane = (uint32_t)lane_id();
  const uint64_t high = uniform64(t.meta[leaf].high), next = uniform64(t.meta[leaf].next);
  const uint32_t count = meta_count(uniform64(t.meta[leaf].info));
  uint64_t k[SPL], v[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const int sl = j * WAVE + (int)lane;
    const size_t at = (size_t)leaf * F + (size_t)min(sl, F - 1);
    const uint64_t kk = t.keys[at];
    v[j] = t.vals[at];
    k[j] = sl < F ? kk : KEY_EMPTY;
  }
  const Spread sp(count + (uint32_t)__popcll(newm), nl, leaf, base);
  // Places in key order: the old entries below plus the new keys below.
  uint32_t r[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) r[j] = 0;
  uint32_t rn = (uint32_t)__popcll(newm & lanemask_lt());
  for (uint32_t i = 0; i < count; ++i) {
    const uint64_t ki = wave_at<F>(k, i);
#pragma unroll
    for (int j = 0; j < SPL; ++j) r[j] += ki < k[j] ? 1u : 0u;
    rn += ki < key ? 1u : 0u;
  }
  for (uint64_t rest = newm; rest; rest &= rest - 1) {
    const uint64_t ki = readlane64(key, __builtin_ctzll(rest));
#pragma unroll
    for (int j = 0; j < SPL; ++j) r[j] += ki < k[j] ? 1u : 0u;
  }
#pragma unroll
  for (int j = 0; j < SPL; ++j)
    if ((uint32_t)(j * WAVE) + lane < count) spread_entry<F>(t, sp, r[j], k[j], v[j]);
  if ((newm >> lane) & 1ull) spread_entry<F>(t, sp, rn, key, val);
  spread_finish<F>(t, sp, 0, count, high, next);
  if (t.rank_of && lane == 0) {
    const uint32_t q = t.rank_of[leaf];
    if (q != NODE_NONE) t.dir[q].pflags |= DIR_SPLIT;
  }
}

// First id of n new inner nodes (after the batch's new leaves; the pool holds them, see the request
// in k_upsert_runs).
STM_DEV uint32_t new_inner(const TreeView& t, SplitState* split, uint32_t n) {
  uint32_t at = 0;
  if (lane_id() == 0) at = atomicAdd(&split->inner, n);
  return (uint32_t)uniform64(t.hdr->n_nodes) + min(uniform32(split->made), uniform32(split->refused)) +
         uniform32(at);
}

// Brings the new children of inner node id (each child's `made`) into it; run by one wavefront.
// A node that overfills is spread over several like a leaf.  Returns whether it was.
template <int F>
STM_DEV bool absorb_children(const TreeView& t, SplitState* split, uint32_t id, TxCounters& c) {
  constexpr int SPL = WNode<F>::SPL;
  const uint32_t lane = (uint32_t)lane_id();
  NodeMeta* m = t.meta + id;
  // Agent-scope loads where an earlier level of the same launch may have written.
  const uint64_t info = uniform64(ld_relaxed(&m->info)), high = uniform64(ld_relaxed(&m->high));
  const uint64_t next = uniform64(ld_relaxed(&m->next));
  const uint32_t count = min(meta_count(info), (uint32_t)F);
  uint64_t k[SPL], v[SPL], made[SPL];
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const int sl = j * WAVE + (int)lane;
    const size_t at = (size_t)id * F + (size_t)min(sl, F - 1);
    k[j] = t.keys[at];
    v[j] = t.vals[at];
  }
  uint32_t r[SPL], total = 0;
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const uint32_t sl = (uint32_t)(j * WAVE) + lane;
    made[j] = sl < count && v[j] < t.capacity ? ld_relaxed(&t.meta[v[j]].made) : 0;
    const uint32_t x = (uint32_t)(made[j] >> 32);
    if (x) st_relaxed(&t.meta[v[j]].made, 0ull);
    uint32_t incl = x;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, WAVE);
      if ((int)lane >= off) incl += y;
    }
    r[j] = sl + total + incl - x;
    total += (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVE - 1);
  }
  if (lane == 0) st_relaxed(&m->dirty, 0ull);
  if (total == 0) return false;
  const uint32_t T = count + total;
  const uint32_t nl = T <= (uint32_t)F ? 1u : spread_nodes<F>(T);
  const Spread sp(T, nl, id, nl > 1 ? new_inner(t, split, nl - 1) : 0u);
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const uint32_t sl = (uint32_t)(j * WAVE) + lane;
    if (sl < count) {
      if (nl > 1 || r[j] != sl) spread_entry<F>(t, sp, r[j], k[j], v[j]);
    }
    // The new children: a lane those of its own child, the whole wavefront where there are many.
    const uint32_t x = (uint32_t)(made[j] >> 32), b = (uint32_t)made[j];
    const bool many = x > 8;
    for (uint32_t q = 0; q < (many ? 0u : x); ++q)
      spread_entry<F>(t, sp, r[j] + 1 + q, ld_relaxed(&t.meta[b + q].low), (uint64_t)(b + q));
    for (uint64_t mm = ballot(many); mm; mm &= mm - 1) {
      const int l = __builtin_ctzll(mm);
      const uint32_t xl = (uint32_t)__builtin_amdgcn_readlane((int)x, l);
      const uint32_t bl = (uint32_t)__builtin_amdgcn_readlane((int)b, l);
      const uint32_t rl = (uint32_t)__builtin_amdgcn_readlane((int)r[j], l);
      for (uint32_t q = lane; q < xl; q += WAVE)
        spread_entry<F>(t, sp, rl + 1 + q, ld_relaxed(&t.meta[bl + q].low), (uint64_t)(bl + q));
    }
  }
  c.node_reads++;
  if (nl == 1) {
    if (lane == 0) st_relaxed(&m->info, make_info(T, meta_level(info)));
    return false;
  }
  spread_finish<F>(t, sp, meta_level(info), count, high, next);
  c.inner_splits += nl - 1;
  c.commits++;
  return true;
}

// Puts inner node id on the list of parents with new children, once.
STM_DEV void list_parent(const TreeView& t, uint32_t id, uint32_t* __restrict__ list, uint32_t* n) {
  if (atomicOr((unsigned long long*)&t.meta[id].dirty, 1ull) == 0) list[atomicAdd(n, 1u)] = id;
}

// Parents of split leaves: one wavefront per level-1 node.  A node that is itself split is listed
// for the level above (k_upsert_finish), by its parent; the root is noted instead.
template <int F>
STM_DEV void absorb_and_list(const TreeView& t, SplitState* split, uint32_t id, uint32_t level,
                             uint32_t* __restrict__ list, uint32_t* n, TxCounters& c) {
  const uint64_t low = uniform64(t.meta[id].low);
  if (!absorb_children<F>(t, split, id, c)) return;
  if ((uint32_t)uniform64(t.hdr->root) == id) {
    if (lane_id() == 0)
      __hip_atomic_store(&split->root, id + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    const uint32_t up = find_at_level<F>(t, low, level + 1);
    if (up != NODE_NONE && lane_id() == 0) list_parent(t, up, list, n);
  }
}

template <int F>
__global__ __launch_bounds__(256) void k_upsert_parents(TreeView t, SplitState* split,
                                                        const uint32_t* __restrict__ plist,
                                                        uint32_t* __restrict__ plist2) {
  const uint32_t n = split->n_dirty;
  const uint32_t nw = gridDim.x * (blockDim.x / WAVE);
  const uint32_t w = uniform32((blockIdx.x * blockDim.x + threadIdx.x) / WAVE);
  if (w >= n) return;
  TxCounters c;
  for (uint32_t i = w; i < n; i += nw)
    absorb_and_list<F>(t, split, uniform32(plist[i]), 1, plist2, &split->n_dirty2, c);
  flush_counters(t, c);
}

// The levels above: one workgroup, level by level (a level lists at most one node per split node
// of the level below, a 48th of them in the mean), then a new root if the root was split.  Takes
// level 1 too when first_level is 1 (few inserts: the list is short and a launch is saved).  Words
// that another wavefront may have written in the same launch are read past the scalar cache.
template <int F>
STM_DEV void upper_pass(const TreeView& t, SplitState* split, uint32_t* plist, uint32_t* plist2,
                        uint32_t first_level) {
  __shared__ uint32_t s_n[2];
  const uint32_t wave = uniform32(threadIdx.x / WAVE);
  if (threadIdx.x == 0) {
    s_n[0] = ld_relaxed32(first_level == 1 ? &split->n_dirty : &split->n_dirty2);
    s_n[1] = 0;
  }
  __syncthreads();
  TxCounters c;
  uint32_t* from = first_level == 1 ? plist : plist2;
  uint32_t* to = first_level == 1 ? plist2 : plist;
  uint32_t cur = 0;
  for (uint32_t level = first_level; level < 64; ++level) {
    const uint32_t n = s_n[cur];
    if (n == 0) break;
    for (uint32_t i = wave; i < n; i += 1024 / WAVE)
      absorb_and_list<F>(t, split, uniform32(ld_relaxed32(from + i)), level, to, &s_n[cur ^ 1], c);
    __syncthreads();  // the level's nodes and the next level's list are written
    if (threadIdx.x == 0) s_n[cur] = 0;
    cur ^= 1;
    uint32_t* x = from;
    from = to;
    to = x;
    __syncthreads();
  }
  __syncthreads();
  if (wave == 0) {
    const uint32_t lane = (uint32_t)lane_id();
    const uint32_t r1 = uniform32(ld_relaxed32(&split->root));
    if (r1) {
      // The split root and its new siblings become the children of a new root, over as many
      // levels as they take (one, unless a batch put tens of thousands of keys into the tree's
      // only leaf).
      uint32_t node = r1 - 1, made = 0;  // the top level: node, then made siblings from base on
      uint32_t base = 0;
      const uint64_t m0 = uniform64(ld_relaxed(&t.meta[node].made));
      base = (uint32_t)m0;
      made = (uint32_t)(m0 >> 32);
      uint32_t level = meta_level(uniform64(ld_relaxed(&t.meta[node].info)));
      while (made) {
        const uint32_t T = made + 1;
        const uint32_t nl = T <= (uint32_t)F ? 1u : spread_nodes<F>(T);
        const uint32_t q = new_inner(t, split, nl);
        const Spread sp(T, nl, q, q + 1);
        level += 1;
        for (uint32_t r = lane; r < T; r += WAVE) {
          const uint32_t child = r == 0 ? node : base + r - 1;
          spread_entry<F>(t, sp, r, r == 0 ? 0ull : ld_relaxed(&t.meta[child].low), (uint64_t)child);
        }
        spread_finish<F>(t, sp, level, (uint32_t)F, KEY_EMPTY, (uint64_t)NODE_NONE);
        if (lane == 0) {
          st_relaxed(&t.meta[q].low, 0ull);
          st_relaxed(&t.meta[q].made, 0ull);
          st_relaxed(&t.meta[node].made, 0ull);
          t.hdr->root = q;
          t.hdr->height = level + 1;
        }
        wave_order();  // the next level reads these nodes' fences
        node = q;
        base = q + 1;
        made = nl - 1;
        c.root_splits++;
      }
    }
    if (lane == 0)
      t.hdr->n_nodes += min(ld_relaxed32(&split->made), ld_relaxed32(&split->refused)) +
                        ld_relaxed32(&split->inner);
  }
  flush_counters(t, c);
}

// New leaves for a request of n: the first id, or NODE_NONE if the pool could not also hold every
// inner node that may follow.  The ids start at the header's n_nodes, which no kernel moves
// before k_upsert_finish.  A split leaves every node at least half full, so new inner nodes number
// at most one per F / 2 - 1 nodes; nor are there more than one per new leaf and level.  By one lane.
template <int F>
STM_DEV uint32_t new_leaves(const TreeView& t, SplitState* split, uint32_t n) {
  const uint32_t at = atomicAdd(&split->made, n);
  const uint64_t nodes = t.hdr->n_nodes, made = (uint64_t)at + n;
  const uint64_t inner = min(made * (t.hdr->height + 1), (nodes + made) / (F / 2 - 1));
  if (nodes + made + inner + 64 <= t.capacity) return (uint32_t)nodes + at;
  atomicMin(&split->refused, at);
  return NODE_NONE;
}

// Exclusive count, over a workgroup of 1024 threads, of the threads with p, and their total.
STM_DEV uint32_t block_rank_1024(bool p, uint32_t* s_w /*[16]*/, uint32_t& total) {
  const uint32_t wave = threadIdx.x / WAVE;
  const uint64_t m = ballot(p);
  if (lane_id() == 0) s_w[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (uint32_t q = 0; q < 1024 / WAVE; ++q) {
    const uint32_t x = s_w[q];
    before += q < wave ? x : 0u;
    total += x;
  }
  __syncthreads();
  return before + (uint32_t)__popcll(m & lanemask_lt());
}

// Number of the n ascending keys below x.
STM_DEV uint32_t count_below(const uint64_t* s, uint32_t n, uint64_t x) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (s[mid] < x) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Runs of more than 64 ops: one workgroup takes a run 1024 ops at a time.  The first pass answers
// the ops, stores the values of keys the leaf holds and counts the new keys; the second merges the
// new keys (in order already) with the leaf's entries by rank and writes each to its place in the
// old leaf or one of the new ones.  As in split_run nothing is locked and the parent learns of the
// new leaves from the next launches.  (Transactions of up to 64 keys each, one after the other
// since they share a leaf, took 20 µs apiece: the first batch of 2^21 ops at 50/50 beside Zipf-hot
// keys, a quarter of its inserts in one leaf, took 75 ms that way and takes 3.1 ms.)
template <int F>
STM_DEV void long_runs(const TreeView& t, const UpsertArgs& a, uint64_t* __restrict__ out_vals,
                       uint8_t* __restrict__ out_found) {
  const uint64_t* __restrict__ ukey = a.ukey;
  const uint64_t* __restrict__ uval = a.uval;
  const uint32_t* __restrict__ sidx = a.sidx;
  const uint32_t* __restrict__ ilist = a.ilist;
  const InsHint* __restrict__ ihint = a.ihint;
  BatchCounters* cnt = a.counters;
  SplitState* split = a.split;
  uint32_t* __restrict__ plist = a.plist;
  uint32_t* __restrict__ dlist = a.dlist;
  constexpr uint32_t BT = 1024;
  __shared__ uint64_t s_raw[F], s_xk[F], s_xv[F];
  __shared__ uint64_t s_new[BT];
  __shared__ uint32_t s_w[BT / WAVE];
  __shared__ uint32_t s_base;
  const uint32_t runs = ld_relaxed32(&split->n_long);
  if (blockIdx.x >= runs) return;
  const uint32_t tid = threadIdx.x;
  const uint32_t wave = uniform32(tid / WAVE);
  TxCounters c;
  uint32_t upserts = 0;
  for (uint32_t q = blockIdx.x; q < runs; q += gridDim.x) {
    const uint32_t e0 = uniform32(ld_relaxed32(a.rlist + q)), len = uniform32(ld_relaxed32(a.rlen + q));
    const InsHint h0 = ihint[ilist[e0]];
    const uint64_t key0 = ukey[ilist[e0]];
    const uint32_t leaf = h0.leaf;
    const uint32_t count = h0.pos >> UPOS_COUNT_SHIFT;
    const size_t nb = (size_t)leaf * F;
    uint32_t news = 0;
    for (uint32_t b = 0; b < len; b += BT) {
      const bool in = b + tid < len;
      const uint32_t gi = ilist[e0 + min(b + tid, len - 1)];
      const InsHint h = ihint[gi];
      const bool found = (h.pos & UPOS_FOUND) != 0;
      const uint32_t p0 = pos_of(sidx[h.gs]);
      uint64_t old = 0;
      if (in && found) {
        const size_t at = nb + (h.pos & UPOS_SLOT);
        old = t.vals[at];
        t.vals[at] = uval[gi];
      }
      write_upsert_answers(in, found, old, h.gs, h.np, p0, sidx, out_vals, out_found);
      uint32_t total;
      (void)block_rank_1024(in && !found, s_w, total);
      news += total;
    }
    const uint32_t T = count + news;
    const uint32_t nl = T <= (uint32_t)F ? 1u : spread_nodes<F>(T);
    if (tid == 0) s_base = nl > 1 ? new_leaves<F>(t, split, nl - 1) : 0u;
    __builtin_amdgcn_s_waitcnt(0);  // the values stored above are read below
    __syncthreads();
    const uint32_t base = s_base;
    const uint64_t high = t.meta[leaf].high, next = t.meta[leaf].next;
    uint64_t xk = 0, xv = 0;
    if (tid < count) {
      xk = t.keys[nb + tid];
      xv = t.vals[nb + tid];
      s_raw[tid] = xk;
    }
    __syncthreads();
    uint32_t xr = 0;  // new keys below the thread's entry
    if (tid < count) {
      uint32_t r = 0;
      for (uint32_t i = 0; i < count; ++i) r += s_raw[i] < xk ? 1u : 0u;
      s_xk[r] = xk;
      s_xv[r] = xv;
    }
    __syncthreads();
    if (tid < count) {
      xk = s_xk[tid];
      xv = s_xv[tid];
    }
    const Spread sp(T, nl, leaf, base);
    uint32_t before = 0;
    for (uint32_t b = 0; b < len; b += BT) {
      const bool in = b + tid < len;
      const uint32_t gi = ilist[e0 + min(b + tid, len - 1)];
      const bool fresh = in && !(ihint[gi].pos & UPOS_FOUND);
      const uint64_t key = ukey[gi], val = uval[gi];
      uint32_t total;
      const uint32_t idx = block_rank_1024(fresh, s_w, total);
      if (base == NODE_NONE) {  // the pool refused: transactions take the keys past a full leaf
        const uint32_t at = count + before + idx;
        if (fresh && at < (uint32_t)F) {
          t.keys[nb + at] = key;
          t.vals[nb + at] = val;
        } else if (fresh) {
          dlist[atomicAdd(&cnt->n_deferred, 1u)] = gi;
        }
        before += total;
        continue;
      }
      if (fresh) s_new[idx] = key;
      __syncthreads();
      if (fresh) spread_entry<F>(t, sp, before + idx + count_below(s_xk, count, key), key, val);
      if (tid < count) xr += count_below(s_new, total, xk);
      before += total;
      __syncthreads();
    }
    if (base != NODE_NONE) {
      if (tid < count) spread_entry<F>(t, sp, tid + xr, xk, xv);
      spread_finish<F>(t, sp, 0, count, high, next, wave, BT / WAVE);
    } else if (tid == 0) {  // (more entries than slots, or no request would have been made)
      st_relaxed(&t.meta[leaf].info, make_info(F, 0));
    }
    __syncthreads();  // LDS is the next run's
    if (wave == 0) {
      upserts += base == NODE_NONE ? len - (T - F) : len;
      c.node_reads += len;
      c.commits++;
      c.new_keys += base == NODE_NONE ? F - count : news;
      if (base != NODE_NONE) c.leaf_splits += nl - 1;
      if (nl > 1 && base != NODE_NONE) {
        uint32_t par = NODE_NONE;
        const uint32_t p = h0.par;
        if (p < t.capacity && meta_level(uniform64(t.meta[p].info)) == 1 &&
            key0 >= uniform64(t.meta[p].low) && key0 < uniform64(t.meta[p].high))
          par = p;
        if (par == NODE_NONE) par = find_at_level<F>(t, key0, 1);
        if (lane_id() == 0) {
          if (par == NODE_NONE) split->root = leaf + 1;  // the leaf is the root
          else list_parent(t, par, plist, &split->n_dirty);
          if (t.rank_of) {
            const uint32_t r = t.rank_of[leaf];
            if (r != NODE_NONE) t.dir[r].pflags |= DIR_SPLIT;
          }
        }
      }
    }
  }
  if (wave == 0) {
    flush_counters(t, c, cnt);
    if (lane_id() == 0) stat_add(t.stats, ST_UPSERTS, blockIdx.x, upserts);
  }
}

// The batch's answer arrays.
struct OutArrays {
  uint64_t* vals;
  uint8_t* found;
};
STM_DEV OutArrays out_arrays(const UpsertArgs& a) {
  return a.desc ? OutArrays{a.desc->out_vals, a.desc->out_found} : OutArrays{a.out_vals, a.out_found};
}

template <int F>
__global__ __launch_bounds__(1024) void k_upsert_long(TreeView t, UpsertArgs a) {
  const OutArrays o = out_arrays(a);
  long_runs<F>(t, a, o.vals, o.found);
}

// The batch's merged INSERTs, one lane per op.  The insert list is in key order,
// so the ops of a leaf are neighbours in it: a run.  A wavefront owns the runs that start in its
// part of the list, and the lanes of a run are the only ones in the launch that touch its leaf, so
// no lock is taken and the lookup kernel's hint (leaf, slot, entry count) is exact: no writer ran
// since.  The r-th new key of a run is appended at slot count + r (a ballot; leaf entries are
// unordered), a present key takes its value in place, and the run's first lane writes the new
// count.  A run that overfills its leaf is split here (split_run) into new leaves that only the
// sibling chain knows; the parents are brought up to date by the next two launches, one
// wavefront per parent, so that the splits under one parent do not queue for its lock.
// Runs too long for a window go to k_upsert_long (split->n_long of them, from the start of rlist and
// rlen).  With piece below 64 (upsert_ops_per_wave: fewer ops per wavefront than a window holds),
// runs of more than `piece` ops go to the transactions of k_upsert instead, cut into pieces of that
// many: wavefront w records them at rlist (first entry) and rlen (ops) from index rfirst[w] on,
// rcount[w] of them; that is the index of the first run it owns, so no two wavefronts' records
// meet.
// Bound by the gathers and scattered stores of an op (its record, key, value, the leaf's slot and
// its answer, each a line of its own), all of which are in flight at once for 64 ops.  In the form
// before, lane groups of eight proved by reading eight earlier groups that an op was the first of
// its leaf, every other op of a leaf took a test-and-set of its lock, and every split a transaction
// through its parent's lock.  Upsert kernels per batch, before / now: 2^22 ops at 95/5 (210 K
// inserts) 73 / 57 µs; 2^19 ops at 50/50 (262 K inserts, most leaves split) 517 / 99 µs; 2^14 ops
// at 50/50 beside Zipf-hot keys 830 / 72 µs.
// Entries of the insert list a wavefront owns at least.  It looks at 64 in any case; owning all of
// them saves reads where the chip is full, but a wavefront splits its overfull leaves one after the
// other, some 4 µs each, so lists of up to RUN_SPREAD_OPS are dealt out in parts of RUN_PART.  16
// batches of 2^14 ops at 50/50 beside Zipf-hot keys, µs: parts of 64 entries 2850, 16 2440, 8 2385; lists of 2^18 in parts of 32 gained nothing.  A list of
// up to 64 stays with one wavefront (1000-op call with 50 inserts 30.0 µs, dealt out 30.3).
constexpr uint32_t RUN_PART = 8;
constexpr uint32_t RUN_SPREAD_OPS = 1u << 16;
template <int F>
STM_DEV void leaf_runs(const TreeView& t, const UpsertArgs& a, uint64_t* __restrict__ out_vals,
                       uint8_t* __restrict__ out_found) {
  const uint64_t* __restrict__ ukey = a.ukey;
  const uint64_t* __restrict__ uval = a.uval;
  const uint32_t* __restrict__ sidx = a.sidx;
  const uint32_t* __restrict__ ilist = a.ilist;
  const InsHint* __restrict__ ihint = a.ihint;
  BatchCounters* cnt = a.counters;
  SplitState* split = a.split;
  uint32_t* __restrict__ plist = a.plist;
  uint32_t* __restrict__ rlist = a.rlist;
  uint32_t* __restrict__ rlen = a.rlen;
  uint32_t* __restrict__ dlist = a.dlist;
  const uint32_t piece = a.piece;
  const uint32_t N = cnt->n_upserts;
  if (a.fanout)
    fanout_answers(a.fanout, a.fanout_cap, cnt, a.gstart, a.npend, a.gval, sidx, out_vals, out_found);
  const uint32_t nw = gridDim.x * (blockDim.x / WAVE);
  const uint32_t w = uniform32((blockIdx.x * blockDim.x + threadIdx.x) / WAVE);
  const uint32_t per = max((N + nw - 1) / nw, N > (uint32_t)WAVE && N <= RUN_SPREAD_OPS ? RUN_PART : (uint32_t)WAVE);
  const uint32_t e0 = (uint32_t)min<uint64_t>((uint64_t)w * per, N);
  const uint32_t e1 = min(e0 + per, N);
  const uint32_t lane = (uint32_t)lane_id();
  const uint64_t lt = lanemask_lt();
  TxCounters c;
  uint32_t upserts = 0;
  uint32_t first = NODE_NONE;  // the first run owned
  uint32_t recs = 0;
  uint32_t base = e0;
  uint32_t left = e0 > 0 && e0 < e1 ? uniform32(entry_leaf(ilist, ihint, e0 - 1)) : NODE_NONE;
  while (base < e1) {
    const uint32_t e = base + lane;
    const bool in = e < N;
    const uint32_t gi = ilist[min(e, N - 1)];
    const uint32_t over = base + WAVE;  // the entry after the window
    const uint32_t gi_over = ilist[min(over, N - 1)];
    const InsHint h = ihint[gi];
    const uint64_t key = ukey[gi];
    const uint64_t val = uval[gi];
    const uint32_t leaf_over = uniform32(ihint[gi_over].leaf);
    const uint32_t p0 = pos_of(sidx[h.gs]);
    const uint32_t leaf = h.leaf;
    const uint32_t up = (uint32_t)__shfl((int)leaf, (int)(lane > 0 ? lane - 1 : 0), WAVE);
    const uint32_t prev = lane > 0 ? up : left;
    const uint64_t hm = ballot(in && (leaf != prev || e == 0));
    const uint32_t last_leaf = (uint32_t)__builtin_amdgcn_readlane((int)leaf, WAVE - 1);
    // The window's last run is whole when the list ends with it or the next entry has another leaf.
    const bool whole = over >= N || leaf_over != last_leaf;
    const uint64_t up_to = hm & (lt | (1ull << lane));
    const uint32_t hl = up_to ? 63u - (uint32_t)__clzll((long long)up_to) : 0u;  // my run's first lane
    const uint64_t above = hm & ~(lt | (1ull << lane));
    const bool is_last = above == 0;
    const uint32_t last_head = hm ? 63u - (uint32_t)__clzll((long long)hm) : 0u;
    if (first == NODE_NONE && hm && base + (uint32_t)__builtin_ctzll(hm) < e1)
      first = base + (uint32_t)__builtin_ctzll(hm);
    // The ops to run now: of a whole run that starts in this wavefront's part.
    const bool mine = in && up_to && base + hl < e1 && (!is_last || whole);
    const uint64_t run = ballot(mine) & (~0ull << hl) &
                         (above ? (above & (0 - above)) - 1 : ~0ull);
    const bool hfound = (h.pos & UPOS_FOUND) != 0;
    const uint32_t slot = h.pos & UPOS_SLOT;
    const uint32_t count = h.pos >> UPOS_COUNT_SHIFT;
    // Hints out of range (never written by the lookup kernel) are not acted on.
    const bool sane = leaf < t.capacity && count <= (uint32_t)F && (!hfound || slot < count);
    const uint64_t badm = ballot(mine && !sane);
    const uint64_t newm = ballot(mine && !hfound) & run;
    const uint32_t news = (uint32_t)__popcll(newm);
    const bool fits = mine && !(badm & run) && count + news <= (uint32_t)F;
    // Overfull runs to split here: new leaves for all of them from one request.
    const uint32_t len = (uint32_t)__popcll(run);
    const uint32_t nl = spread_nodes<F>(count + news);
    const uint32_t want = mine && !fits && !(badm & run) && len <= piece && lane == hl ? nl - 1 : 0u;
    uint64_t splitm = ballot(want != 0);
    uint32_t nb0 = 0;  // first new leaf of the run (its first lane)
    if (splitm) {
      uint32_t incl = want;
#pragma unroll
      for (int off = 1; off < WAVE; off <<= 1) {
        const uint32_t y = __shfl_up(incl, off, WAVE);
        if ((int)lane >= off) incl += y;
      }
      const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, WAVE - 1);
      uint32_t at = 0;
      if (lane == 0) at = new_leaves<F>(t, split, total);
      at = uniform32(at);
      if (at == NODE_NONE) splitm = 0;
      nb0 = at + incl - want;
    }
    const bool splits = mine && ((splitm >> hl) & 1ull);
    // A run that the pool refused: what needs no node is done here, up to a full leaf.
    const bool refused = mine && !fits && !splits && !(badm & run) && piece >= (uint32_t)WAVE;
    const bool placed = fits || splits || refused;
    const size_t nb = (size_t)(placed ? leaf : 0u) * F;
    const uint32_t at = count + (uint32_t)__popcll(newm & lt);  // of a new key
    const bool answered = fits || splits || (refused && (hfound || at < (uint32_t)F));
    uint64_t old = 0;
    if (answered) {
      if (hfound) {
        old = t.vals[nb + slot];
        t.vals[nb + slot] = val;
      } else if (!splits) {
        t.keys[nb + at] = key;
        t.vals[nb + at] = val;
      }
    }
    if (placed && !splits && lane == hl && news)
      st_relaxed(&t.meta[leaf].info, make_info(min(count + news, (uint32_t)F), 0));
    write_upsert_answers(answered, hfound, old, h.gs, h.np, p0, sidx, out_vals, out_found);
    const uint64_t okm = ballot(answered);
    c.commits += (uint32_t)__popcll(okm & hm);
    c.new_keys += (uint32_t)__popcll(ballot(answered && !hfound));
    c.node_reads += (uint32_t)__popcll(okm);
    upserts += (uint32_t)__popcll(okm);
    if (splitm) {
      wave_order();  // the values above are in place before the leaves are read
      // The parents, by every run's first lane at once: the level-1 node the lookup kernel routed
      // through when its fences hold the key, else by a descent below.
      uint32_t par = NODE_NONE;
      if ((splitm >> lane) & 1ull) {
        const uint32_t p = h.par;
        const NodeMeta* pm = t.meta + (p < t.capacity ? p : 0u);
        const uint64_t pinfo = pm->info, plow = pm->low, phigh = pm->high;
        if (p < t.capacity && meta_level(pinfo) == 1 && key >= plow && key < phigh) par = p;
      }
      for (uint64_t sm = splitm; sm; sm &= sm - 1) {
        const int l = __builtin_ctzll(sm);
        const uint32_t lf = (uint32_t)__builtin_amdgcn_readlane((int)leaf, l);
        const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)nl, l);
        split_run<F>(t, lf, (uint32_t)__builtin_amdgcn_readlane((int)nb0, l), n, readlane64(newm, l),
                     key, val);
        c.leaf_splits += n - 1;
        if ((uint32_t)__builtin_amdgcn_readlane((int)par, l) == NODE_NONE) {
          const uint32_t p = find_at_level<F>(t, readlane64(key, l), 1);
          if (p == NODE_NONE) {  // the leaf is the root
            if (lane == 0) split->root = lf + 1;
          } else if ((int)lane == l) {
            par = p;
          }
        }
      }
      if (par != NODE_NONE) list_parent(t, par, plist, &split->n_dirty);
    }
    // A run that did not fit its leaf as it is: the attempt in place is given up and the run done
    // again (a split here, or by one of the kernels after this one).
    const uint64_t again = ballot(mine && !fits);
    c.aborts += (uint32_t)__popcll(again & hm);
    const uint64_t leave = ballot(mine && !answered);
    if (piece >= (uint32_t)WAVE) {
      // Refused by the pool, for want of a node (or a hint out of range): transactions at the end.
      if (leave) {
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&cnt->n_deferred, (uint32_t)__popcll(leave));
        at = uniform32(at);
        if ((leave >> lane) & 1ull) dlist[at + (uint32_t)__popcll(leave & lt)] = gi;
      }
    } else {
      for (uint64_t lm = leave & hm; lm; lm &= lm - 1) {
        const int l = __builtin_ctzll(lm);
        const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)len, l);
        const uint32_t pieces = (n + piece - 1) / piece;
        if (lane < pieces) {
          rlist[first + recs + lane] = base + (uint32_t)l + lane * piece;
          rlen[first + recs + lane] = min(piece, n - lane * piece);
        }
        recs += pieces;
      }
    }
    uint32_t next;  // lane of the first entry not dealt with (WAVE: the next window)
    if (hm == 0 || whole || base + last_head >= e1) {
      next = WAVE;
    } else if (last_head > 0) {
      next = last_head;
    } else {
      // A run longer than the window.
      const uint32_t end = run_end(ilist, ihint, base + WAVE - 1, N, last_leaf);
      const uint32_t n = end - base;
      c.aborts++;
      if (piece >= (uint32_t)WAVE) {
        if (lane == 0) {
          const uint32_t at = atomicAdd(&split->n_long, 1u);
          rlist[at] = base;
          rlen[at] = n;
        }
      } else {
        const uint32_t pieces = (n + piece - 1) / piece;
        for (uint32_t q = lane; q < pieces; q += WAVE) {
          rlist[first + recs + q] = base + q * piece;
          rlen[first + recs + q] = min(piece, n - q * piece);
        }
        recs += pieces;
      }
      left = last_leaf;
      base = end;
      continue;
    }
    left = (uint32_t)__builtin_amdgcn_readlane((int)leaf, (int)next - 1);
    base += next;
  }
  if (lane == 0) {
    a.rfirst[w] = first;
    a.rcount[w] = recs;
  }
  flush_counters(t, c, cnt);
  if (lane == 0) stat_add(t.stats, ST_UPSERTS, wave_stripe(), upserts);
}

template <int F>
__global__ __launch_bounds__(256) void k_upsert_runs(TreeView t, UpsertArgs a) {
  const OutArrays o = out_arrays(a);
  leaf_runs<F>(t, a, o.vals, o.found);
}

// Wave-wide transactions for a round of ops, group gi per lane with `mine`.  Ops of the round whose
// keys share a leaf commit together (tx_merge_attempt): a hot leaf takes one transaction per round
// instead of one per op.  Ops that exhaust their attempts go to `later` (*n_later of them).
template <int F>
STM_DEV void tx_ops(const TreeView& t, const UpsertArgs& a, uint32_t gi, bool mine,
                    uint64_t* __restrict__ out_vals, uint8_t* __restrict__ out_found,
                    uint32_t* later, uint32_t* n_later, TxCounters& c, ParentCache<F>& pc,
                    uint32_t& upserts, uint32_t& deferred) {
  // The round's op data, loaded together and read lane by lane.
  uint64_t todo = ballot(mine);
  const InsHint h = a.ihint[gi];
  const uint64_t k_l = a.ukey[gi];
  const uint64_t v_l = a.uval[gi];
  const uint32_t gs_l = h.gs, np_l = h.np, par_l = h.par, leaf_l = h.leaf;
  const uint32_t p0_l = pos_of(a.sidx[gs_l]);
  while (todo) {
    const int l = __builtin_ctzll(todo);
    const uint64_t key = readlane64(k_l, l);
    const uint32_t ph = __builtin_amdgcn_readlane(par_l, l);
    const uint32_t lh = __builtin_amdgcn_readlane(leaf_l, l);
    uint32_t aborts = 0, restarts = 0;
    uint64_t done = 0;
    bool found_l = false;
    uint64_t old_l = 0;
    bool gave_up = false;
    for (;;) {
      // The hint is only tried on the first attempt; retries descend from the root.
      const bool first = aborts + restarts == 0;
      const TxResult r = tx_merge_attempt<F>(t, key, todo, k_l, v_l, c, pc,
                                             first ? ph : NODE_NONE, first ? lh : NODE_NONE,
                                             done, found_l, old_l);
      if (r == TX_DONE) break;
      if (r == TX_FAIL) {  // pool exhausted: error bit raised, the op is dropped
        done = 1ull << l;
        found_l = false;
        old_l = 0;
        break;
      }
      if (r == TX_ABORT) {
        c.aborts++;
        if (++aborts >= a.max_attempts) {
          gave_up = true;
          break;
        }
        backoff(aborts);
      } else if (++restarts >= 4 * a.max_attempts) {  // TX_RESTART after a preemptive split
        gave_up = true;
        break;
      }
    }
    if (gave_up) {  // the op of lane l goes to the serial pass
      const uint32_t g = __builtin_amdgcn_readlane(gi, l);
      if (lane_id() == 0)
        __hip_atomic_store(later + atomicAdd(n_later, 1u), g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      deferred++;
      upserts++;
      todo &= ~(1ull << l);
      continue;
    }
    write_upsert_answers(((done >> lane_id()) & 1ull) != 0, found_l, old_l, gs_l, np_l, p0_l, a.sidx,
                         out_vals, out_found);
    upserts += (uint32_t)__popcll(done);
    todo &= ~done;
  }
}

// The runs that k_upsert_runs left for transactions: many inserts into one leaf.
// Wavefront f of that kernel recorded rcount[f] pieces from index rfirst[f] of rlist / rlen on.
// With r = nw / run_waves wavefronts here per wavefront there, each takes every r-th of its pieces;
// with fewer, wavefront w takes all pieces of wavefronts w, w + nw, ...  A piece is the ops of one
// leaf in key order, so the ops of a round mostly commit in one transaction, and only the parent is
// shared with other wavefronts (and the leaf, when its run was cut into pieces).
template <int F>
__global__ __launch_bounds__(256) void k_upsert(TreeView t, UpsertArgs a, uint32_t run_waves) {
  BatchCounters* cnt = a.counters;
  if (cnt->n_upserts == 0) return;
  const OutArrays o = out_arrays(a);
  const uint32_t nw = gridDim.x * (blockDim.x / WAVE);
  const uint32_t w = uniform32((blockIdx.x * blockDim.x + threadIdx.x) / WAVE);
  const uint32_t r = max(nw / run_waves, 1u);
  TxCounters c;
  ParentCache<F> pc;
  uint32_t upserts = 0, deferred = 0;
  for (uint32_t f = w / r; f < run_waves; f += nw / r) {
    const uint32_t pieces = uniform32(a.rcount[f]);
    const uint32_t at = uniform32(a.rfirst[f]);
    for (uint32_t q = w % r; q < pieces; q += r) {
      const uint32_t s0 = uniform32(a.rlist[at + q]);
      const uint32_t s1 = s0 + uniform32(a.rlen[at + q]);
      for (uint32_t base = s0; base < s1; base += WAVE) {
        const uint32_t e = base + lane_id();
        tx_ops<F>(t, a, a.ilist[min(e, s1 - 1)], e < s1, o.vals, o.found, a.dlist, &cnt->n_deferred, c,
                  pc, upserts, deferred);
      }
    }
  }
  flush_counters(t, c, cnt);
  if (lane_id() == 0) {
    stat_add(t.stats, ST_UPSERTS, wave_stripe(), upserts);
    stat_add(t.stats, ST_DEFERRED, wave_stripe(), deferred);
  }
}

// The n ops of the runs that the all but full pool refused, in dlist: a wavefront takes 64 at a
// time (they were listed run by run, so the ops of a leaf are mostly together).
template <int F>
STM_DEV void refused_ops(const TreeView& t, const UpsertArgs& a, uint32_t n,
                         uint64_t* __restrict__ out_vals, uint8_t* __restrict__ out_found) {
  TxCounters c;
  ParentCache<F> pc;
  uint32_t upserts = 0, deferred = 0;
  for (;;) {
    uint32_t at = 0;
    if (lane_id() == 0) at = atomicAdd(&a.split->head, (uint32_t)WAVE);
    at = uniform32(at);
    if (at >= n) break;
    const uint32_t e = at + lane_id();
    tx_ops<F>(t, a, ld_relaxed32(a.dlist + min(e, n - 1)), e < n, out_vals, out_found, a.rlist,
              &a.split->n_redo, c, pc, upserts, deferred);
  }
  flush_counters(t, c, a.counters);
  if (lane_id() == 0) {
    stat_add(t.stats, ST_UPSERTS, wave_stripe(), upserts);
    stat_add(t.stats, ST_DEFERRED, wave_stripe(), deferred);
  }
}

// The batch's counters and the tree's error bits: lane l below 8 holds 64-bit word l of the block.
// Agent-scope loads see the other kernels' and wavefronts' updates past this CU's cache.
struct CounterWords {
  uint64_t w, err;
  STM_DEV uint32_t at(size_t offset) const {
    const uint64_t x = readlane64(w, (int)(offset / 8));
    return (uint32_t)(offset % 8 ? x >> 32 : x);
  }
};
static_assert(sizeof(BatchCounters) == 64 && offsetof(BatchCounters, hdr_error) == 40,
              "hdr_error is word 5");
STM_DEV CounterWords load_counters(const TreeView& t, const BatchCounters* cnt) {
  return CounterWords{ld_relaxed(reinterpret_cast<const uint64_t*>(cnt) + (lane_id() & 7)),
                      ld_relaxed(&t.hdr->error)};
}

// Serial pass over the n ops of `list`, which exhausted their attempts: one wavefront, no
// competitors, so every transaction commits on its first attempt.  Then the batch's counters.
template <int F>
STM_DEV void serial_pass(const TreeView& t, const UpsertArgs& a, CounterWords cw, const uint32_t* list,
                         uint32_t n, uint64_t* __restrict__ out_vals,
                         uint8_t* __restrict__ out_found) {
  BatchCounters* cnt = a.counters;
  if (n) {
    TxCounters c;
    ParentCache<F> pc;
    for (uint32_t e = 0; e < n; ++e) {
      const uint32_t g = uniform32(ld_relaxed32(list + e));
      if (!run_upsert<F>(t, a.ukey[g], a.uval[g], a.gstart[g], a.npend[g], a.sidx, out_vals, out_found,
                         1024u, c, pc)) {
        if (lane_id() == 0) atomicOr((unsigned long long*)&t.hdr->error, (unsigned long long)ERR_LIVELOCK);
      }
    }
    flush_counters(t, c, cnt);
    wave_order();
    cw = load_counters(t, cnt);
  }
  // The last kernel of a batch: the tree's error bits travel back with the batch counters.
  const uint32_t skipped = cw.at(offsetof(BatchCounters, skipped));
  const uint32_t retry = cw.at(offsetof(BatchCounters, sort_retry));
  const uint32_t unique = cw.at(offsetof(BatchCounters, n_unique));
  const uint32_t bad = cw.at(offsetof(BatchCounters, n_bad));
  const uint32_t stall = cw.at(offsetof(BatchCounters, sort_stall));
  const uint32_t fallback = cw.at(offsetof(BatchCounters, sort_fallback));
  const uint32_t splits = cw.at(offsetof(BatchCounters, leaf_splits));
  if (lane_id() == 0) {
    cnt->hdr_error = cw.err;
    if (StreamAcc* acc = a.acc) {
      if (skipped) {
        acc->skipped += 1;
      } else if (retry) {  // ran empty: the host runs it again and resumes the stream after it
        acc->retries += 1;
      } else {
        acc->unique += unique;
        acc->bad += bad;
        acc->sort_stalls += stall;
        acc->fallbacks += fallback;
        acc->leaf_splits += splits;
        acc->batches += 1;
      }
    }
  }
  if (a.host_counters) {
    // Lanes 0-7 store the 64-byte block into pinned host memory, which spares the batch a
    // separate copy on the stream; the system fence makes the stores visible before the kernel ends.
    const int l = lane_id();
    if (l < 8)
      __hip_atomic_store(reinterpret_cast<uint64_t*>(a.host_counters) + l, l == 5 ? cw.err : cw.w,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
  }
}

// The end of a batch's upserts: one workgroup brings the upper levels of the tree up to date, the
// ops that the pool refused run as transactions, and one wavefront does the serial pass and the
// counters.  A batch of at most ONE_BLOCK_OPS ops has its leaf runs, short and long, done here
// too.  Each phase sees the writes of the ones before: every wavefront has its stores acknowledged
// before the barrier, and the words they share are read past the scalar cache.
// A small batch pays for launches and round trips: what the phases need to know (long runs, splits,
// refused ops, counters) comes in one.  As four launches (runs, long runs, upper levels, serial
// pass) a 1000-op call took 33.3 µs, as one 29.5; with the upper levels and the serial pass in one
// launch a 40001-op call takes 81 µs instead of 84.  Above ONE_BLOCK_OPS one workgroup would take its
// runs in turns: the grid of k_upsert_runs takes them at once.
// Only a pool that is all but full refuses runs, and then tens of thousands of ops at once may wait
// for transactions, which the other workgroups of the grid are for (they leave at once otherwise).
// Those wait, for a bounded time, until the first has the upper levels done; the ops are dealt out
// from a counter, so a workgroup that gave up is not missed.  The last to arrive goes on alone.
constexpr uint32_t FIN_RUNS = 1, FIN_UPPER = 2, FIN_SERIAL = 4;
constexpr uint32_t FIN_BLOCKS = 32;
constexpr uint32_t UPPER_POLLS = 1u << 18;  // of 64 clocks of sleep and a load each
template <int F, uint32_t PHASES>
__global__ __launch_bounds__(1024) void k_upsert_finish(TreeView t, UpsertArgs a, uint32_t first_level) {
  __shared__ uint32_t s_flag;
  const OutArrays o = out_arrays(a);
  SplitState* split = a.split;
  if constexpr ((PHASES & FIN_RUNS) != 0) {  // (one workgroup)
    leaf_runs<F>(t, a, o.vals, o.found);
    wave_order();
    __syncthreads();
  }
  const uint32_t n_long = PHASES & FIN_RUNS ? ld_relaxed32(&split->n_long) : 0u;
  uint32_t made = ld_relaxed32(&split->made);
  CounterWords cw = load_counters(t, a.counters);
  uint32_t listed = cw.at(offsetof(BatchCounters, n_deferred));  // in dlist
  bool changed = false;
  if ((PHASES & FIN_RUNS) && n_long) {
    long_runs<F>(t, a, o.vals, o.found);
    wave_order();
    __syncthreads();
    made = ld_relaxed32(&split->made);
    listed = ld_relaxed32(&a.counters->n_deferred);
    changed = true;
  }
  bool go = true;
  if (blockIdx.x > 0) {
    if (listed == 0) return;
    if (threadIdx.x == 0) {
      uint32_t done = 0;
      for (uint32_t p = 0; !done && p < UPPER_POLLS; ++p) {
        done = ld_relaxed32(&split->upper);
        if (!done) __builtin_amdgcn_s_sleep(1);
      }
      s_flag = done;
    }
    __syncthreads();
    go = s_flag != 0;
  } else if ((PHASES & FIN_UPPER) && made) {
    upper_pass<F>(t, split, a.plist, a.plist2, first_level);
    wave_order();
    __syncthreads();
    changed = true;
  }
  const uint32_t* list = a.dlist;
  if ((PHASES & FIN_UPPER) && (PHASES & FIN_SERIAL) && listed) {
    if (blockIdx.x == 0) {
      // The nodes' plain stores leave this XCD's cache before the transactions read them.
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __syncthreads();
      if (threadIdx.x == 0)
        __hip_atomic_store(&split->upper, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (go) refused_ops<F>(t, a, listed, o.vals, o.found);
    wave_order();
    __syncthreads();
    if (gridDim.x > 1) {
      if (threadIdx.x == 0) s_flag = atomicAdd(&split->arrived, 1u) + 1 == gridDim.x;
      __syncthreads();
      if (!s_flag) return;
    }
    list = a.rlist;
    listed = ld_relaxed32(&split->n_redo);
    changed = true;
  }
  if ((PHASES & FIN_SERIAL) && threadIdx.x < (uint32_t)WAVE) {
    if (changed) cw = load_counters(t, a.counters);
    serial_pass<F>(t, a, cw, list, listed, o.vals, o.found);
  }
}

// ================================================================== dump / check
__global__ void k_collect_leaves(TreeView t, uint32_t n_nodes, uint64_t* __restrict__ lows,
                                 uint32_t* __restrict__ ids, uint32_t* __restrict__ counter) {
  const uint32_t id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= n_nodes) return;
  const NodeMeta m = t.meta[id];
  if (meta_level(m.info) != 0) return;
  const uint32_t slot = atomicAdd(counter, 1u);
  lows[slot] = m.low;
  ids[slot] = id;
}

__global__ void k_leaf_counts(TreeView t, const uint32_t* __restrict__ order,
                              const uint32_t* __restrict__ ids_unsorted, uint32_t n_leaves,
                              uint32_t* __restrict__ sorted_ids, uint32_t* __restrict__ counts) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_leaves) return;
  const uint32_t id = ids_unsorted[order[r]];
  sorted_ids[r] = id;
  counts[r] = meta_count(t.meta[id].info);
}

template <int F>
__global__ void k_dump_copy(TreeView t, const uint32_t* __restrict__ sorted_ids,
                            const uint64_t* __restrict__ offsets, uint32_t n_leaves,
                            uint64_t* __restrict__ out_k, uint64_t* __restrict__ out_v) {
  const uint64_t gi = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
  if (gi >= (uint64_t)n_leaves * F) return;
  const uint32_t r = (uint32_t)(gi / F);
  const uint32_t s = (uint32_t)(gi % F);
  const uint64_t o0 = offsets[r];
  const uint64_t o1 = offsets[r + 1];
  if (o0 + s >= o1) return;
  const uint32_t id = sorted_ids[r];
  // A leaf's entries are unordered: slot s goes to its rank among the leaf's count entries.
  const uint64_t* kp = t.keys + (size_t)id * F;
  const uint64_t k = kp[s];
  const uint32_t count = (uint32_t)(o1 - o0);
  uint32_t rank = 0;
  for (uint32_t u = 0; u < count; ++u) rank += kp[u] < k ? 1u : 0u;
  out_k[o0 + rank] = k;
  out_v[o0 + rank] = t.vals[(size_t)id * F + s];
}

// One wavefront per node; counts violated invariants into *bad.
template <int F>
__global__ __launch_bounds__(256) void k_check(TreeView t, uint32_t n_nodes,
                                               unsigned long long* bad) {
  constexpr int SPL = WNode<F>::SPL;
  const uint32_t id = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
  if (id >= n_nodes) return;
  const NodeMeta m = t.meta[id];
  const uint32_t count = meta_count(m.info);
  const uint32_t level = meta_level(m.info);
  uint32_t errs = 0;
  if (m.lock & 1) errs++;
  if (count > (uint32_t)F) {
    if (lane_id() == 0) atomicAdd(bad, 1ull);
    return;
  }
  if (m.low >= m.high) errs++;
#pragma unroll
  for (int j = 0; j < SPL; ++j) {
    const int s = j * WAVE + lane_id();
    if (s >= F) continue;
    const uint64_t k = t.keys[(size_t)id * F + s];
    const uint64_t v = t.vals[(size_t)id * F + s];
    if ((uint32_t)s >= count) {
      if (k != KEY_EMPTY) errs++;
      continue;
    }
    if (level > 0) {
      if (s > 0 && t.keys[(size_t)id * F + s - 1] >= k) errs++;  // inner nodes in key order
    } else {
      // leaf entries are unordered but distinct
      for (uint32_t u = 0; u < count; ++u)
        if (u != (uint32_t)s && t.keys[(size_t)id * F + u] == k) errs++;
    }
    if (k < m.low || k >= m.high) errs++;
    if (level > 0) {
      if (s == 0 && k != m.low) errs++;
      if (v >= n_nodes) {
        errs++;
        continue;
      }
      const NodeMeta cm = t.meta[v];
      if (meta_level(cm.info) + 1 != level) errs++;
      if (cm.low != k) errs++;
      const uint64_t hi = ((uint32_t)s + 1 < count) ? t.keys[(size_t)id * F + s + 1] : m.high;
      if (cm.high != hi) errs++;
    }
  }
  if (lane_id() == 0) {
    if (m.next != NODE_NONE) {
      if (m.next >= n_nodes) errs++;
      else {
        const NodeMeta nm = t.meta[m.next];
        if (nm.low != m.high || meta_level(nm.info) != level) errs++;
      }
    } else if (m.high != KEY_EMPTY) {
      errs++;
    }
    if (level > 0 && count == 0) errs++;
  }
  for (int off = 32; off >= 1; off >>= 1) errs += __shfl_xor(errs, off, WAVE);
  if (lane_id() == 0 && errs) atomicAdd(bad, (unsigned long long)errs);
}

// ================================================================== launchers
template <int F>
static hipError_t launch_build_leaves_f(const TreeView& t, const uint64_t* ukey, const uint64_t* uval,
                                        uint32_t U, uint32_t fill, uint32_t L, uint64_t* lows,
                                        hipStream_t s) {
  const uint64_t n = (uint64_t)L * F;
  k_build_leaves<F><<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(t, ukey, uval, U, fill, L, lows);
  return hipGetLastError();
}
template <int F>
static hipError_t launch_build_inner_f(const TreeView& t, const uint64_t* lows_prev, uint32_t n_prev,
                                       uint32_t first_prev, uint32_t fill, uint32_t n_this,
                                       uint32_t first_this, uint32_t level, uint64_t* lows_out,
                                       hipStream_t s) {
  const uint64_t n = (uint64_t)n_this * F;
  k_build_inner<F><<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(t, lows_prev, n_prev, first_prev, fill,
                                                               n_this, first_this, level, lows_out);
  return hipGetLastError();
}

#define STM_DISPATCH_F(F_, CALL)   \
  switch (F_) {                    \
    case 32: { constexpr int F = 32; return CALL; } \
    case 64: { constexpr int F = 64; return CALL; } \
    case 128: { constexpr int F = 128; return CALL; } \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_build_leaves(const TreeView& t, const uint64_t* ukey, const uint64_t* uval,
                               uint32_t U, uint32_t fill, uint32_t L, uint64_t* lows, hipStream_t s) {
  STM_DISPATCH_F(t.fanout, launch_build_leaves_f<F>(t, ukey, uval, U, fill, L, lows, s));
}
hipError_t launch_build_inner(const TreeView& t, const uint64_t* lows_prev, uint32_t n_prev,
                              uint32_t first_prev, uint32_t fill, uint32_t n_this,
                              uint32_t first_this, uint32_t level, uint64_t* lows_out,
                              hipStream_t s) {
  STM_DISPATCH_F(t.fanout, launch_build_inner_f<F>(t, lows_prev, n_prev, first_prev, fill, n_this,
                                                   first_this, level, lows_out, s));
}

// Lane groups of a lookup kernel the device holds at once (asked once per instantiation).
template <int F, int G, bool LEARNED, bool INDEX>
static hipError_t lookup_fill(uint32_t& fill) {
  static std::atomic<uint32_t> groups{0};
  uint32_t v = groups.load(std::memory_order_relaxed);
  if (v == 0) {
    int dev = 0, cus = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
      e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_lookup<F, G, LEARNED, INDEX>, 256, 0);
    if (e != hipSuccess) return e;
    v = (uint32_t)std::max(1, cus * per_cu) * (256u / G);
    groups.store(v, std::memory_order_relaxed);
  }
  fill = v;
  return hipSuccess;
}

template <int F, int G, bool LEARNED, bool INDEX>
static hipError_t launch_lookup_k(const TreeView& t, const LookupArgs& a, hipStream_t s) {
  uint32_t fill = 1;
  hipError_t e = lookup_fill<F, G, LEARNED, INDEX>(fill);
  if (e != hipSuccess) return e;
  // A lane group per chunk of ops, but never fewer groups than ops or than the device holds at
  // once: a lane group's ops are a chain of dependent node reads, so a small batch that gave each
  // group a whole chunk ran sixteen chains' length on a mostly idle device (whole call at 1000 ops
  // 112 -> 85 µs, at 40001 ops 165 -> 149 µs; from chunk * fill ops, 458752 at 16 lanes and
  // chunks of 16, the spans are what they were).
  const uint64_t groups = std::max<uint64_t>((a.n_max + a.chunk - 1) / a.chunk,
                                             std::min<uint64_t>(a.n_max, fill));
  // Persistent grid: at most LOOKUP_GRID_CAP workgroups; each lane group walks one contiguous span.
  const uint32_t blocks = (uint32_t)std::min<uint64_t>((groups * G + 255) / 256, LOOKUP_GRID_CAP);
  if (blocks == 0) return hipSuccess;
  k_lookup<F, G, LEARNED, INDEX><<<blocks, 256, 0, s>>>(
      t, a.ukey, a.uop, a.gstart, a.npend, a.sidx, a.counters, a.chunk, fill, a.out_vals,
      a.out_found, LEARNED ? a.route_hdr : nullptr, LEARNED ? a.fences : nullptr,
      LEARNED ? a.lids : nullptr, LEARNED ? a.segs : nullptr, a.desc, a.ihint, a.gval, a.fanout,
      a.fanout_cap, a.split, a.acc);
  return hipGetLastError();
}

template <int F, int G>
static hipError_t launch_lookup_fg(const TreeView& t, const LookupArgs& a, hipStream_t s) {
  if (a.route_hdr && a.index) return launch_lookup_k<F, G, true, true>(t, a, s);
  if (a.route_hdr) return launch_lookup_k<F, G, true, false>(t, a, s);
  return launch_lookup_k<F, G, false, false>(t, a, s);
}

template <int F>
static hipError_t launch_lookup_f(const TreeView& t, const LookupArgs& a, hipStream_t s) {
  switch (a.lanes) {
    case 8: return launch_lookup_fg<F, 8>(t, a, s);
    case 16: return launch_lookup_fg<F, 16>(t, a, s);
    case 32: return launch_lookup_fg<F, (F >= 32 ? 32 : 16)>(t, a, s);
    case 64: return launch_lookup_fg<F, (F >= 64 ? 64 : 32)>(t, a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_lookup(const TreeView& t, const LookupArgs& a, hipStream_t s) {
  STM_DISPATCH_F(t.fanout, launch_lookup_f<F>(t, a, s));
}

template <int F>
static hipError_t launch_upsert_f(const TreeView& t, const UpsertArgs& a, hipStream_t s) {
  // Each wavefront takes an equal contiguous share of the merged INSERTs, at least 64 of them (8 of
  // a short list): a grid of at most the wavefronts the chip holds at once works through them in one
  // generation.
  static std::atomic<int> resident{0};  // blocks of this instantiation the device holds at once
  if (resident.load(std::memory_order_relaxed) == 0) {
    int dev = 0, cus = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess)
      e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_upsert_runs<F>, 256, 0);
    if (e != hipSuccess) return e;
    resident.store(std::max(1, cus * per_cu), std::memory_order_relaxed);
  }
  const uint32_t blocks = std::min<uint32_t>(
      std::min<uint32_t>((uint32_t)((a.n_max + 63) / 64), (uint32_t)resident.load(std::memory_order_relaxed)),
      RUN_WAVES_MAX / 4);
  const uint32_t waves = blocks * 4;  // one rfirst / rcount entry per wavefront
  const bool runs_only = a.piece >= (uint32_t)WAVE;
  hipError_t e;
  if (runs_only && a.n_max <= ONE_BLOCK_OPS) {
    k_upsert_finish<F, FIN_RUNS | FIN_UPPER | FIN_SERIAL><<<1, 1024, 0, s>>>(t, a, 1u);
    return hipGetLastError();
  }
  k_upsert_runs<F><<<blocks, 256, 0, s>>>(t, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (runs_only) {
    const uint32_t lb = std::min<uint32_t>((uint32_t)(a.n_max / WAVE), LONG_BLOCKS);
    if (lb > 0) {  // no run of more than 64 ops in fewer
      k_upsert_long<F><<<lb, 1024, 0, s>>>(t, a);
      if ((e = hipGetLastError()) != hipSuccess) return e;
    }
  }
  const bool few = a.n_max <= FEW_INSERTS;
  if (!few) {
    k_upsert_parents<F><<<PARENT_BLOCKS, 256, 0, s>>>(t, a.split, a.plist, a.plist2);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  const uint32_t first_level = few ? 1u : 2u;
  if (runs_only) {
    const uint32_t fb = std::max<uint32_t>(1, std::min<uint32_t>((uint32_t)(a.n_max / 1024), FIN_BLOCKS));
    k_upsert_finish<F, FIN_UPPER | FIN_SERIAL><<<fb, 1024, 0, s>>>(t, a, first_level);
    return hipGetLastError();
  }
  k_upsert_finish<F, FIN_UPPER><<<1, 1024, 0, s>>>(t, a, first_level);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  k_upsert<F><<<a.blocks, 256, 0, s>>>(t, a, waves);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  k_upsert_finish<F, FIN_SERIAL><<<1, 64, 0, s>>>(t, a, first_level);
  return hipGetLastError();
}

hipError_t launch_upsert(const TreeView& t, const UpsertArgs& a, hipStream_t s) {
  STM_DISPATCH_F(t.fanout, launch_upsert_f<F>(t, a, s));
}

hipError_t launch_collect_leaves(const TreeView& t, uint32_t n_nodes, uint64_t* lows, uint32_t* ids,
                                 uint32_t* counter, hipStream_t s) {
  if (n_nodes == 0) return hipSuccess;
  k_collect_leaves<<<(n_nodes + 255) / 256, 256, 0, s>>>(t, n_nodes, lows, ids, counter);
  return hipGetLastError();
}
hipError_t launch_leaf_counts(const TreeView& t, const uint32_t* order, const uint32_t* ids,
                              uint32_t n_leaves, uint32_t* sorted_ids, uint32_t* counts,
                              hipStream_t s) {
  if (n_leaves == 0) return hipSuccess;
  k_leaf_counts<<<(n_leaves + 255) / 256, 256, 0, s>>>(t, order, ids, n_leaves, sorted_ids, counts);
  return hipGetLastError();
}
template <int F>
static hipError_t launch_dump_copy_f(const TreeView& t, const uint32_t* sorted_ids,
                                     const uint64_t* offsets, uint32_t n_leaves, uint64_t* out_k,
                                     uint64_t* out_v, hipStream_t s) {
  const uint64_t n = (uint64_t)n_leaves * F;
  if (n == 0) return hipSuccess;
  k_dump_copy<F><<<(uint32_t)((n + 255) / 256), 256, 0, s>>>(t, sorted_ids, offsets, n_leaves, out_k, out_v);
  return hipGetLastError();
}
hipError_t launch_dump_copy(const TreeView& t, const uint32_t* sorted_ids, const uint64_t* offsets,
                            uint32_t n_leaves, uint64_t* out_k, uint64_t* out_v, hipStream_t s) {
  STM_DISPATCH_F(t.fanout, launch_dump_copy_f<F>(t, sorted_ids, offsets, n_leaves, out_k, out_v, s));
}
template <int F>
static hipError_t launch_check_f(const TreeView& t, uint32_t n_nodes, unsigned long long* bad,
                                 hipStream_t s) {
  if (n_nodes == 0) return hipSuccess;
  const uint64_t threads = (uint64_t)n_nodes * WAVE;
  k_check<F><<<(uint32_t)((threads + 255) / 256), 256, 0, s>>>(t, n_nodes, bad);
  return hipGetLastError();
}
hipError_t launch_check(const TreeView& t, uint32_t n_nodes, unsigned long long* bad, hipStream_t s) {
  STM_DISPATCH_F(t.fanout, launch_check_f<F>(t, n_nodes, bad, s));
}

}  // namespace stm
