// stm_api.hip — the C ABI of include/stmtree.h: tree object, batch pipeline, bulk build,
// dump, structural check and statistics.
//
// Batch pipeline on the tree's stream (reference: GPU_STM_Tree::gpu_work_main,
// src/gpu-stm-tree-v38/bpt-gpustm.cpp:77-167, and launchKernelBefore/launchKernel/
// launchKernelAfter, src/gpu-stm-tree-v38/bpt-gpustm-kernel.cu:264-332):
//   sort (key, position)  ->  per-key fold  ->  read-only lookups  ->  transactional upserts
// Batches longer than max_batch are cut into consecutive chunks, as the reference cuts
// its input file into batch_size pieces; each chunk completes before the next starts,
// so results do not depend on the chunking.  No host round trip happens inside a chunk
// (the reference copies the run count to the host between RLE and scan, :303).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/stmtree.h"
#include "stm_common.hpp"
#include "stm_internal.hpp"
#include "stm_pairs.hpp"
#include "stm_tree.hpp"

using namespace stm;

namespace {

thread_local std::string g_last_error;

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

#define HIP_TRY(expr)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess)                                                                \
      return fail(e_ == hipErrorOutOfMemory ? STM_ERR_NOMEM : STM_ERR_DEVICE, "%s: %s (%s:%d)", \
                  #expr, hipGetErrorString(e_), __FILE__, __LINE__);                     \
  } while (0)

template <typename T>
hipError_t dalloc(T** p, size_t count) {
  *p = nullptr;
  if (count == 0) count = 1;
  return hipMalloc((void**)p, count * sizeof(T));
}

constexpr uint32_t DESC_TABLE = 4096;  // descriptors uploaded per window of a stream
constexpr int GRAPH_CLASSES = 12;      // size classes 2^10, 2^12, ..., up to max_batch
constexpr uint32_t GRAPH_MAX_OPS = 1u << 12;  // classes that are captured
constexpr uint32_t OVERLAP_MIN_OPS = 2049;    // batches whose front half may run on its own stream
constexpr uint64_t OVERLAP_BATCHES = 32;      // such batches before that stream is made

// Waits, for at most a tenth of a millisecond, until k_probe_set has run; says whether it saw it.
__global__ void k_probe_wait(uint32_t* flag, uint32_t* seen) {
  if (threadIdx.x != 0) return;
  const uint64_t until = wall_clock64() + 10000;  // 100 MHz
  while (!__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
    if (wall_clock64() > until) return;
    __builtin_amdgcn_s_sleep(4);
  }
  *seen = 1;
}
__global__ void k_probe_set(uint32_t* flag) {
  if (threadIdx.x == 0)
    __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// First node of every replayed graph: takes the next descriptor of the window.
__global__ void k_advance(const BatchDesc* __restrict__ table, uint32_t* __restrict__ cursor,
                          BatchDesc* __restrict__ live) {
  if (threadIdx.x != 0) return;
  const uint32_t c = cursor[0];
  *live = table[c];
  cursor[0] = c + 1;
}

// Plain streaming copy of n16 16-byte words: the known-size reference kernel for HBM traffic
// counters and the measured bandwidth ceiling.  One word per thread over a grid that covers the
// whole copy: on gfx950 this outruns both a resident grid-stride loop and several words in
// flight per thread (6.2 TB/s read + write against 4.7-5.6 TB/s at 4 GiB).  The stride loop
// only serves copies beyond COPY_MAX_BLOCKS blocks.
constexpr uint32_t COPY_MAX_BLOCKS = 1u << 24;
__global__ __launch_bounds__(256) void k_copy16(uint4* __restrict__ dst, const uint4* __restrict__ src,
                                                uint64_t n16) {
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * 256ull)
    dst[i] = src[i];
}

// Where an array of a slab goes: arrays lie back to back, 256-byte aligned.  One allocation holds
// them all (a tree has about sixty arrays; each hipMalloc and hipFree of its own cost 10-300 µs,
// 12 of the 17 ms that creating, loading, using and closing a tree of 2^20 keys took).
struct SlabCursor {
  uint8_t* base;  // null: only count
  size_t at = 0;
  void* take(size_t bytes) {
    at = (at + 255) / 256 * 256;
    void* p = base ? base + at : nullptr;
    at += std::max<size_t>(bytes, 1);
    return p;
  }
};

struct Scratch {
  uint64_t n = 0;
  void* slab = nullptr;  // the allocation that holds every device array (null: a fixed region does)
  uint64_t *in_keys = nullptr, *in_vals = nullptr, *out_vals = nullptr;
  uint8_t *in_ops = nullptr, *out_found = nullptr;
  uint64_t *skeys_tmp = nullptr, *skeys = nullptr;
  uint32_t *sidx_tmp = nullptr, *sidx = nullptr;
  uint32_t* hist = nullptr;
  uint32_t* front = nullptr;  // front half of small batches (front_scratch_words)
  void* fold_tiles = nullptr;
  uint64_t *ukey = nullptr, *uval = nullptr;
  uint8_t* uop = nullptr;
  uint32_t *gstart = nullptr, *npend = nullptr, *dlist = nullptr;
  uint32_t *rlist = nullptr, *rlen = nullptr;  // pieces of runs that need a split (UpsertArgs)
  uint32_t *rfirst = nullptr, *rcount = nullptr;  // per wavefront of k_upsert_runs
  SplitState* split = nullptr;  // leaves split without a lock, and the parents to update
  uint32_t *plist = nullptr, *plist2 = nullptr;
  uint32_t* ilist = nullptr;  // merged INSERTs of the batch, in key order
  InsHint* ihint = nullptr;   // the lookup kernel's record of every merged INSERT
  uint64_t* fanout = nullptr; // answer chunks of hot GET groups (fanout_capacity(n))
  BatchCounters* counters = nullptr;
  BatchCounters* h_counters = nullptr;  // pinned host copy for the per-batch readback
  // range scans
  uint64_t *soff = nullptr, *scan_tiles = nullptr;
  int32_t* lastins = nullptr;
  // batch streams replayed from captured graphs
  BatchDesc* desc_table = nullptr;  // DESC_TABLE entries
  BatchDesc* desc_live = nullptr;   // the batch the current replay works on
  uint32_t* cursor = nullptr;       // next desc_table entry
  StreamAcc* acc = nullptr;

  // What a scratch is for: a tree's synchronous calls (host staging and stream control too), the
  // second set of a batch stream, or one bulk load (sort and fold only).
  enum Use { CALLS, STREAM, LOAD };

  // Every device array of the scratch for batches of up to cap ops, in one fixed order.
  void layout(uint64_t cap, Use use, SlabCursor& cur) {
    n = cap;
#define A_(p, c) p = static_cast<decltype(p)>(cur.take(sizeof(*p) * (size_t)(c)))
    const bool staging = use == CALLS;
    if (use != LOAD) A_(in_ops, cap);
    if (staging) {
      A_(in_keys, cap); A_(in_vals, cap); A_(out_vals, cap); A_(out_found, cap);
    }
    A_(skeys_tmp, cap); A_(skeys, cap); A_(sidx_tmp, cap); A_(sidx, cap);
    A_(hist, sort_hist_words(cap));
    A_(front, front_scratch_words());
    uint8_t* ft = nullptr;
    A_(ft, fold_scratch_bytes(cap));
    fold_tiles = ft;
    A_(ukey, cap); A_(uval, cap); A_(uop, cap);
    A_(counters, 1);
    if (use == LOAD) return;
    A_(gstart, cap); A_(npend, cap);
    A_(dlist, cap);
    A_(ihint, cap);
    A_(rlist, cap); A_(rlen, cap);
    A_(rfirst, RUN_WAVES_MAX); A_(rcount, RUN_WAVES_MAX);
    A_(split, 1); A_(plist, cap); A_(plist2, cap);
    A_(ilist, cap);
    A_(fanout, fanout_capacity(cap));
    A_(desc_live, 1);
    if (staging) {
      A_(desc_table, DESC_TABLE); A_(cursor, 1); A_(acc, 1);
      A_(soff, cap); A_(lastins, cap); A_(scan_tiles, scan_tile_words(cap));
    }
#undef A_
  }

  hipError_t alloc(uint64_t cap, Use use) {
    SlabCursor size{nullptr};
    layout(cap, use, size);
    hipError_t e = hipMalloc(&slab, size.at);
    if (e != hipSuccess) {
      *this = Scratch();
      return e;
    }
    SlabCursor place{static_cast<uint8_t*>(slab)};
    layout(cap, use, place);
    if ((e = sort_scratch_init(hist)) != hipSuccess || use != CALLS) return e;
    return hipHostMalloc((void**)&h_counters, sizeof(BatchCounters), hipHostMallocCoherent);
  }

  // Lays the arrays out from base (a fixed region); with base null only counts.  Returns the bytes
  // the layout spans.
  size_t carve(uint64_t cap, uint8_t* base) {
    SlabCursor cur{base};
    layout(cap, STREAM, cur);
    return cur.at;
  }
  void release() {
    if (slab) (void)hipFree(slab);
    if (h_counters) (void)hipHostFree(h_counters);
    *this = Scratch();
  }
};

}  // namespace

struct stm_tree {
  stm_config cfg{};
  hipStream_t stream = nullptr;
  TreeView view{};
  void* pool = nullptr;  // the allocation behind view's arrays
  uint64_t capacity = 0;
  Scratch scr;
  stm_stats st{};
  hipEvent_t ev_a[STM_NUM_PHASES] = {};
  hipEvent_t ev_b[STM_NUM_PHASES] = {};
  hipEvent_t ev_begin[STM_NUM_PHASES] = {};  // the event a phase's time starts from
  bool phase_used[STM_NUM_PHASES] = {};
  // learned routing
  RouteState route;
  void* route_slab = nullptr;  // the allocation behind route's arrays
  bool route_alloc = false;
  bool route_valid = false;       // directory + model describe a recent tree
  bool route_warm = false;        // the segment models were trained on this tree
  uint32_t batches_since_train = 0;
  uint64_t splits_since_train = 0;  // leaf splits counted since the last directory rebuild
  uint64_t dir_leaves = 0;          // leaves of the directory at the last rebuild
  // Batch streams (stm_run_batches_device) run each batch as two halves, on two scratch sets, so
  // that the front half (sort, fold) of batch i + 1 runs on stream_front while the back half
  // (lookups, upserts, counters) of batch i runs on `stream`.  Captured graphs, one per small size
  // class, hold both halves for `stream`.
  Scratch scr2;
  bool scr2_alloc = false;
  hipStream_t stream_front = nullptr;
  hipEvent_t ev_open = nullptr;  // what was queued on `stream` before the stream of batches
  hipEvent_t ev_front[2] = {};  // front half of the set's latest batch done
  hipEvent_t ev_back[2] = {};   // the set's latest batch done (its scratch is free)
  uint64_t overlap_batches = 0;  // batches seen that could have overlapped
  bool pipeline_failed = false;  // and that nothing of this could be made for
  hipGraphExec_t graphs[GRAPH_CLASSES] = {};
  // Batches above 2^18 ops outside the sample sort's sizes sort normalized keys unless exact_left > 0:
  // a batch whose normalized sort had to fall back (long buckets of distinct keys: hot keys with
  // neighbours) makes the next EXACT_HOLD batches use the eight exact passes directly.  (A sample
  // that misled says nothing of the next batch.)  A batch up to 2^18 ops is sorted by the
  // front half's own sort unless front_hold > 0: one that overflowed a bucket there makes the next
  // EXACT_HOLD of them use the exact passes too (launched, not replayed: the captured graphs hold
  // the front half's sort).
  uint32_t exact_left = 0;
  uint32_t front_hold = 0;
  uint64_t sort_fallbacks = 0;  // batches sorted again with the exact passes (stm_stats)
};

namespace {

constexpr uint32_t EXACT_HOLD = 16;

uint64_t capacity_for(uint64_t max_keys, uint32_t F) {
  const uint64_t half = F / 2;
  uint64_t leaves = (max_keys + half - 1) / half + 1;
  uint64_t cap = leaves + leaves / (half - 1) + 64;
  cap += cap / 10 + 1024;
  return cap;
}

int set_device(stm_tree* t) {
  HIP_TRY(hipSetDevice(t->cfg.device));
  return STM_OK;
}

void phase_begin(stm_tree* t, int p) {
  if (!t->cfg.timing) return;
  (void)hipEventRecord(t->ev_a[p], t->stream);
  t->ev_begin[p] = t->ev_a[p];
}
void phase_end(stm_tree* t, int p) {
  if (!t->cfg.timing) return;
  (void)hipEventRecord(t->ev_b[p], t->stream);
  t->phase_used[p] = true;
}
// Phase `from` ends where phase `to` begins: one event marks both.  Each recorded event sits
// between two kernels and holds the second back by a few microseconds, so a boundary costs one
// event instead of two.
void phase_switch(stm_tree* t, int from, int to) {
  if (!t->cfg.timing) return;
  phase_end(t, from);
  t->ev_begin[to] = t->ev_b[from];
}
void phase_collect(stm_tree* t) {
  if (!t->cfg.timing) return;
  for (int p = 0; p < STM_NUM_PHASES; ++p) {
    if (!t->phase_used[p]) continue;
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, t->ev_begin[p], t->ev_b[p]) == hipSuccess) {
      t->st.phase_ms[p] += ms;
      t->st.phase_launches[p] += 1;
    }
    t->phase_used[p] = false;
  }
}

// Sum of the stripes of every device counter (the stream is synchronised first).
int read_counters(stm_tree* t, uint64_t out[ST_NUM]) {
  std::vector<unsigned long long> c(STATS_WORDS);
  HIP_TRY(hipStreamSynchronize(t->stream));
  HIP_TRY(hipMemcpy(c.data(), t->view.stats, sizeof(unsigned long long) * STATS_WORDS,
                    hipMemcpyDeviceToHost));
  for (int k = 0; k < ST_NUM; ++k) {
    uint64_t v = 0;
    for (int j = 0; j < STAT_STRIPES; ++j) v += c[(size_t)k * STAT_STRIPES + j];
    out[k] = v;
  }
  return STM_OK;
}

int read_header(stm_tree* t, TreeHeader* h) {
  HIP_TRY(hipMemcpyAsync(h, t->view.hdr, sizeof(TreeHeader), hipMemcpyDeviceToHost, t->stream));
  HIP_TRY(hipStreamSynchronize(t->stream));
  return STM_OK;
}

int error_bits_status(stm_tree* t, uint64_t error) {
  if (error & ERR_POOL_FULL)
    return fail(STM_ERR_NOMEM, "node pool exhausted (capacity %llu nodes); raise max_keys",
                (unsigned long long)t->capacity);
  if (error & ERR_LIVELOCK) return fail(STM_ERR_DEVICE, "serial upsert pass could not commit");
  return STM_OK;
}

int check_device_error(stm_tree* t) {
  TreeHeader h;
  int rc = read_header(t, &h);
  if (rc) return rc;
  return error_bits_status(t, h.error);
}

// Writes an empty tree: one empty leaf as root.
int init_empty(stm_tree* t) {
  NodeMeta m{};
  m.lock = 0;
  m.info = 0;
  m.low = 0;
  m.high = KEY_EMPTY;
  m.next = NODE_NONE;
  HIP_TRY(hipMemsetAsync(t->view.keys, 0xff, sizeof(uint64_t) * t->cfg.fanout, t->stream));
  HIP_TRY(hipMemsetAsync(t->view.vals, 0, sizeof(uint64_t) * t->cfg.fanout, t->stream));
  HIP_TRY(hipMemcpyAsync(t->view.meta, &m, sizeof(m), hipMemcpyHostToDevice, t->stream));
  TreeHeader h{};
  h.lock = 0;
  h.root = 0;
  h.height = 1;
  h.n_nodes = 1;
  h.capacity = t->capacity;
  h.error = 0;
  h.n_keys = 0;
  HIP_TRY(hipMemcpyAsync(t->view.hdr, &h, sizeof(h), hipMemcpyHostToDevice, t->stream));
  HIP_TRY(hipStreamSynchronize(t->stream));
  return STM_OK;
}

void drop_graphs(stm_tree* t) {
  for (hipGraphExec_t& g : t->graphs) {
    if (g) (void)hipGraphExecDestroy(g);
    g = nullptr;
  }
}

int alloc_router(stm_tree* t) {
  if (t->route_alloc) return STM_OK;
  RouteState& r = t->route;
  const uint64_t cap = t->capacity;
  auto layout = [&](SlabCursor& cur) {
#define A_(p, c) p = static_cast<decltype(p)>(cur.take(sizeof(*p) * (size_t)(c)))
    A_(r.hdr, 1); A_(r.fences, cap + 1); A_(r.lids, cap); A_(r.segs, ROUTE_SEGMENTS);
    A_(r.dir, cap + 1); A_(r.rank_of, cap); A_(r.lows, cap); A_(r.lows_tmp, cap);
    A_(r.sorted_lows, cap); A_(r.order, cap); A_(r.order_tmp, cap); A_(r.hist, sort_hist_words(cap));
    A_(r.dir_alt, cap + 1);
#undef A_
  };
  SlabCursor size{nullptr};
  layout(size);
  if (hipMalloc(&t->route_slab, size.at) != hipSuccess) {
    t->route_slab = nullptr;
    return fail(STM_ERR_NOMEM, "learned-routing buffers for %llu nodes", (unsigned long long)cap);
  }
  SlabCursor place{static_cast<uint8_t*>(t->route_slab)};
  layout(place);
  if (sort_scratch_init(r.hist) != hipSuccess) return fail(STM_ERR_DEVICE, "learned-routing sort scratch");
  t->route_alloc = true;
  t->view.rank_of = r.rank_of;
  t->view.dir = r.dir;
  drop_graphs(t);  // captured with the previous TreeView
  return STM_OK;
}

void free_router(stm_tree* t) {
  if (t->route_slab) (void)hipFree(t->route_slab);
  t->route_slab = nullptr;
  t->route = RouteState();
  t->view.rank_of = nullptr;
  t->view.dir = nullptr;
  t->route_alloc = false;
  t->route_valid = false;
  t->route_warm = false;
}

// Rebuilds the leaf directory from the tree and trains the router (phase "train").  A
// periodic retrain of models already trained on this tree starts from their parameters and
// runs an eighth of the steps (at least 16): a few batches move few leaves.
int train_router(stm_tree* t, uint32_t steps, bool periodic) {
  int rc = alloc_router(t);
  if (rc) return rc;
  TreeHeader h;
  rc = read_header(t, &h);
  if (rc) return rc;
  const uint32_t nn = (uint32_t)std::min<uint64_t>(h.n_nodes, t->capacity);
  const bool index = t->cfg.route == STM_ROUTE_INDEX;
  const bool warm = periodic && t->route_warm;
  // A periodic retrain fine-tunes the converged segment models over the rewritten directory:
  // a few Adam steps (9 of the default 300).  At 2^26 Gamma keys and 2^22-op batches, 37 steps
  // kept 91% of lookups in the predicted window and 9 keep 84%, with the same lookup time (a
  // sorted span reuses its leaf, and a missed window costs one more window read), while the
  // training time per retrain drops by three quarters.
  if (warm) steps = std::max<uint32_t>(steps / 32, 8);
  if (index) steps = 0;  // the static index only needs the directory
  // Adam's first steps move every parameter by about the learning rate whatever the
  // gradient's size, so fine-tuning a converged model uses a tenth of it.
  const float lr = warm ? 0.002f : 0.02f;
  phase_begin(t, STM_PHASE_TRAIN);
  HIP_TRY(route_build(t->view, t->route, nn, steps, lr, steps > 0, warm, t->stream));
  t->route_warm = steps > 0 || index;
  phase_end(t, STM_PHASE_TRAIN);
  if (t->cfg.timing) {  // every retrain is counted, also between graph replays
    HIP_TRY(hipStreamSynchronize(t->stream));
    phase_collect(t);
  }
  t->route_valid = true;
  t->batches_since_train = 0;
  t->splits_since_train = 0;
  RouteHeader rh{};
  HIP_TRY(hipMemcpyAsync(&rh, t->route.hdr, sizeof(rh), hipMemcpyDeviceToHost, t->stream));
  HIP_TRY(hipStreamSynchronize(t->stream));
  t->dir_leaves = rh.L;
  return STM_OK;
}

// The launch sequence of one batch: sort -> fold -> lookups -> upserts.  With in.desc the
// batch (its arrays and its length, at most in.n) is read on the device, which is what a
// captured graph replays; otherwise in.n and the pointers describe it.  No host round trip.
struct PipeIn {
  const uint64_t* keys;
  const uint64_t* vals;
  const uint8_t* ops;
  uint32_t n;
  uint64_t* out_vals;
  uint8_t* out_found;
  const BatchDesc* desc;
  // scan mode: op 3 is SCAN(key, L = vals[i]) with output into scan_keys / scan_vals
  bool scans;
  uint64_t* scan_keys;
  uint64_t* scan_vals;
  uint64_t scan_cap;
  // optional: the last upsert kernel copies the batch counters here (pinned host memory)
  BatchCounters* host_counters;
  // optional: the batch of a stream: runs empty after a failed one, its counters are added here
  StreamAcc* acc;
};

// Front half of a batch: sort and fold.  Reads only the batch and writes only the scratch and
// the outputs of ops the fold answers, never the tree, so it may run on `st` beside the back
// half of the previous batch (on another scratch).
hipError_t enqueue_front(stm_tree* t, Scratch& s, const PipeIn& in, bool timed, bool exact,
                         hipStream_t st) {
  hipError_t e;
  if (timed) phase_begin(t, STM_PHASE_SORT);
  FoldArgs fa{};
  fa.skeys = s.skeys;
  fa.sidx = s.sidx;
  fa.vals = in.vals;
  fa.ops = in.ops;
  fa.n = in.n;
  fa.desc = in.desc;
  fa.out_vals = in.out_vals;
  fa.out_found = in.out_found;
  fa.ukey = s.ukey;
  fa.uval = s.uval;
  fa.uop = s.uop;
  fa.gstart = s.gstart;
  fa.npend = s.npend;
  fa.counters = s.counters;
  fa.tile_scratch = s.fold_tiles;
  fa.lastins = in.scans ? s.lastins : nullptr;
  fa.ilist = s.ilist;
  if (in.n <= FRONT_MAX_OPS && !exact) {
    const FrontArgs fr{in.keys, in.ops, fa, s.skeys_tmp, s.sidx_tmp, s.front};
    if ((e = front_batch(fr, st)) != hipSuccess) return e;
    if (timed) {  // sort and fold in one phase
      phase_switch(t, STM_PHASE_SORT, STM_PHASE_MERGE);
      phase_switch(t, STM_PHASE_MERGE, STM_PHASE_LOOKUP);
    }
    return hipSuccess;
  }
  e = radix_sort_pairs_desc(in.keys, in.ops, in.desc, in.n, s.skeys_tmp, s.skeys, s.sidx_tmp, s.sidx, 0,
                            64, s.hist, (int)t->cfg.sort_tile_items, exact, in.out_found, st);
  if (e != hipSuccess) return e;
  if (timed) phase_switch(t, STM_PHASE_SORT, STM_PHASE_MERGE);
  fa.sort_stall = sort_stall_word(s.hist);
  fa.sort_exact = sort_exact_word(s.hist);
  if ((e = fold_batch(fa, st)) != hipSuccess) return e;
  if (timed) phase_switch(t, STM_PHASE_MERGE, STM_PHASE_LOOKUP);
  return hipSuccess;
}

// Back half: lookups, scans, upserts (and the counters' copy to the host when asked), on the
// tree's stream.
hipError_t enqueue_back(stm_tree* t, Scratch& s, const PipeIn& in, bool timed) {
  hipStream_t st = t->stream;
  hipError_t e;
  ScanArgs sa{};
  if (in.scans) {
    sa.keys = in.keys;
    sa.vals = in.vals;
    sa.ops = in.ops;
    sa.n = in.n;
    sa.desc = in.desc;
    sa.out_vals = in.out_vals;
    sa.out_found = in.out_found;
    sa.scan_keys = in.scan_keys;
    sa.scan_vals = in.scan_vals;
    sa.scan_cap = in.scan_cap;
    sa.ukey = s.ukey;
    sa.uop = s.uop;
    sa.gstart = s.gstart;
    sa.npend = s.npend;
    sa.sidx = s.sidx;
    sa.lastins = s.lastins;
    sa.counters = s.counters;
    sa.soff = s.soff;
    sa.tile_sums = s.scan_tiles;
  }

  LookupArgs la{};
  if (t->cfg.route != STM_ROUTE_DESCENT) {
    la.route_hdr = t->route.hdr;
    la.fences = t->route.fences;
    la.lids = t->route.lids;
    la.segs = t->route.segs;
    la.index = t->cfg.route == STM_ROUTE_INDEX ? 1u : 0u;
  }
  la.ukey = s.ukey;
  la.uop = s.uop;
  la.gstart = s.gstart;
  la.npend = s.npend;
  la.sidx = s.sidx;
  la.counters = s.counters;
  la.n_max = in.n;
  la.chunk = t->cfg.ops_per_group;
  la.lanes = t->cfg.lanes_per_op;
  la.out_vals = in.out_vals;
  la.out_found = in.out_found;
  la.desc = in.desc;
  la.ihint = s.ihint;
  la.gval = s.uval;  // GET groups carry no merged value: a hot group's value goes there
  la.fanout = s.fanout;
  la.fanout_cap = fanout_capacity(in.n);
  la.split = s.split;
  la.acc = in.acc;
  if ((e = launch_lookup(t->view, la, st)) != hipSuccess) return e;

  if (in.scans) {  // on the tree as it was before the batch: before the upsert kernel
    if (timed) phase_switch(t, STM_PHASE_LOOKUP, STM_PHASE_SCAN);
    if ((e = launch_scan_offsets(sa, st)) != hipSuccess) return e;
    if ((e = launch_range_scan(t->view, sa, st)) != hipSuccess) return e;
    if (timed) phase_switch(t, STM_PHASE_SCAN, STM_PHASE_UPSERT);
  } else if (timed) {
    phase_switch(t, STM_PHASE_LOOKUP, STM_PHASE_UPSERT);
  }

  UpsertArgs ua{};
  ua.ukey = s.ukey;
  ua.uval = s.uval;
  ua.gstart = s.gstart;
  ua.npend = s.npend;
  ua.sidx = s.sidx;
  ua.counters = s.counters;
  ua.dlist = s.dlist;
  ua.max_attempts = t->cfg.max_attempts;
  // The transactions' grid: upsert_ops_per_wave batch ops per wavefront, at most 8192 wavefronts
  // (every SIMD of the chip fully occupied).
  const uint64_t waves = ((uint64_t)in.n + t->cfg.upsert_ops_per_wave - 1) / t->cfg.upsert_ops_per_wave;
  ua.blocks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((waves + 3) / 4, 2048));
  ua.out_vals = in.out_vals;
  ua.out_found = in.out_found;
  ua.desc = in.desc;
  ua.ihint = s.ihint;
  ua.ilist = s.ilist;
  ua.n_max = in.n;
  ua.piece = t->cfg.upsert_ops_per_wave;
  ua.split = s.split;
  ua.plist = s.plist;
  ua.plist2 = s.plist2;
  ua.rlist = s.rlist;
  ua.rlen = s.rlen;
  ua.rfirst = s.rfirst;
  ua.rcount = s.rcount;
  ua.fanout = s.fanout;
  ua.fanout_cap = fanout_capacity(in.n);
  ua.gval = s.uval;
  ua.host_counters = in.host_counters;
  ua.acc = in.acc;
  if ((e = launch_upsert(t->view, ua, st)) != hipSuccess) return e;
  if (timed) phase_end(t, STM_PHASE_UPSERT);
  if (in.scans && (e = launch_scan_answers(sa, st)) != hipSuccess) return e;
  return hipSuccess;
}

hipError_t enqueue_pipeline(stm_tree* t, Scratch& s, const PipeIn& in, bool timed, bool exact) {
  hipError_t e = enqueue_front(t, s, in, timed, exact, t->stream);
  if (e != hipSuccess) return e;
  return enqueue_back(t, s, in, timed);
}

// Learned routing and the static index: (re)build the directory, and retrain, when it is
// missing or stale.
// Also after split-heavy batches: once the leaves split since the last rebuild reach
// retrain_splits (a 32nd of the directory's leaves by default), lookups would walk right
// siblings from too many stale entries.
int maybe_retrain(stm_tree* t) {
  if (t->cfg.route == STM_ROUTE_DESCENT) return STM_OK;
  const uint64_t split_limit =
      t->cfg.retrain_splits ? t->cfg.retrain_splits : std::max<uint64_t>(1, t->dir_leaves / 32);
  if (t->route_valid && t->batches_since_train < t->cfg.retrain_every &&
      t->splits_since_train < split_limit)
    return STM_OK;
  return train_router(t, t->cfg.train_steps, true);
}

// Whether found flags and op codes of n ops share memory.
bool overlaps(const uint8_t* found, const uint8_t* ops, size_t n) {
  return found < ops + n && ops < found + n;
}

// Scan output area of a chunk (device pointers); null = op 3 runs as GET.
struct ScanOut {
  uint64_t* keys;
  uint64_t* vals;
  uint64_t cap;
  uint64_t used;  // set by run_chunk: the sum of the chunk's scan lengths
};

// One chunk of at most max_batch ops, all pointers on the device; waits for its completion.
// The batch scratch is the tree's own unless `scr` points at another layout of it.
int run_chunk(stm_tree* t, const uint64_t* keys, const uint64_t* vals, const uint8_t* ops,
              uint32_t n, uint64_t* out_vals, uint8_t* out_found, ScanOut* so = nullptr,
              Scratch* scr = nullptr) {
  Scratch& s = scr ? *scr : t->scr;
  hipStream_t st = t->stream;
  int rc = maybe_retrain(t);
  if (rc) return rc;
  PipeIn in{keys, vals, ops, n, out_vals, out_found, nullptr, false, nullptr, nullptr, 0, nullptr, nullptr};
  if (so) {
    in.scans = true;
    in.scan_keys = so->keys;
    in.scan_vals = so->vals;
    in.scan_cap = so->cap;
  } else {
    in.host_counters = s.h_counters;  // the scan answers kernel runs after the upsert kernels
  }
  if (overlaps(out_found, ops, n)) {  // the flags' default is written before the last look at the ops
    HIP_TRY(hipMemcpyAsync(s.in_ops, ops, n, hipMemcpyDeviceToDevice, st));
    in.ops = s.in_ops;
  }
  const bool small = n <= FRONT_MAX_OPS;
  uint32_t& hold = small ? t->front_hold : t->exact_left;
  const bool sampled = sample_sorted(n);
  bool exact = hold > 0 && !sampled;
  BatchCounters bc;
  for (;;) {
    HIP_TRY(enqueue_pipeline(t, s, in, true, exact));
    // One readback per batch, into pinned memory: counters and the tree's error bits.
    if (so)
      HIP_TRY(hipMemcpyAsync(s.h_counters, s.counters, sizeof(BatchCounters), hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    bc = *s.h_counters;
    if (!bc.sort_retry || exact) break;
    // The small-batch sort overflowed a bucket and the batch ran empty: once more, exactly.
    exact = true;
    hold = EXACT_HOLD + 1;  // this batch and the next EXACT_HOLD
    t->sort_fallbacks += 1;
  }
  phase_collect(t);
  if (bc.sort_stall) return fail(STM_ERR_DEVICE, "batch sort: a grid-barrier wait gave up");
  if (bc.sort_fallback) {
    if (!sampled) t->exact_left = EXACT_HOLD;
    t->sort_fallbacks += 1;
  } else if (exact) {
    hold -= 1;
  }
  t->st.batches += 1;
  t->st.ops += n;
  t->st.unique_ops += bc.n_unique;
  t->batches_since_train += 1;
  t->splits_since_train += bc.leaf_splits;
  if (bc.n_bad) return fail(STM_ERR_INVALID, "batch holds the reserved key 0xffffffffffffffff");
  if (so) {
    so->used = bc.scan_total;
    if (bc.scan_bad)
      return fail(STM_ERR_INVALID, "%u scan ops have a length outside [1, %u] or overflow the "
                  "scan output area (%llu pairs)", bc.scan_bad, SCAN_MAX_LEN,
                  (unsigned long long)so->cap);
  }
  return error_bits_status(t, bc.hdr_error);
}

// ------------------------------------------------------------------ graph replay of streams
uint32_t class_nmax(const stm_tree* t, int c) {
  const uint64_t v = 1024ull << (2 * c);
  return (uint32_t)std::min<uint64_t>(v, t->cfg.max_batch);
}

int class_of(const stm_tree* t, uint32_t n) {
  for (int c = 0; c < GRAPH_CLASSES; ++c)
    if (class_nmax(t, c) >= n) return c;
  return GRAPH_CLASSES - 1;  // max_batch <= 2^30 fits class 10
}

// A stream whose kernels run beside those of `beside`.  Streams share a few hardware queues, and
// two streams on one queue run one after the other (a stream of 2^16-op batches then took 65 µs per
// batch instead of 54), so a candidate is tried: does its kernel reach a kernel that waits on
// `beside`?  The rejected ones are kept until the choice is made, so that each candidate gets another
// queue.
hipError_t stream_beside(hipStream_t beside, uint32_t* words /*2, device*/, hipStream_t* out) {
  constexpr int TRIES = 4;
  hipStream_t tried[TRIES] = {};
  hipError_t e = hipSuccess;
  int n = 0;
  uint32_t seen = 0;
  while (n < TRIES && !seen && e == hipSuccess) {
    if ((e = hipStreamCreate(&tried[n])) != hipSuccess) break;
    hipStream_t c = tried[n++];
    if ((e = hipMemsetAsync(words, 0, 8, beside)) != hipSuccess ||
        (e = hipStreamSynchronize(beside)) != hipSuccess)
      break;
    k_probe_wait<<<1, 64, 0, beside>>>(words, words + 1);
    k_probe_set<<<1, 64, 0, c>>>(words);
    if ((e = hipGetLastError()) != hipSuccess || (e = hipStreamSynchronize(c)) != hipSuccess) break;
    e = hipMemcpyAsync(&seen, words + 1, 4, hipMemcpyDeviceToHost, beside);
    if (e == hipSuccess) e = hipStreamSynchronize(beside);
  }
  const int keep = e == hipSuccess ? n - 1 : -1;
  for (int i = 0; i < n; ++i)
    if (i != keep && tried[i]) (void)hipStreamDestroy(tried[i]);
  if (keep >= 0) *out = tried[keep];
  return e;
}

// The second scratch set, the front stream and the pipeline's events.
hipError_t make_pipeline(stm_tree* t) {
  if (t->scr2_alloc) return hipSuccess;
  hipError_t e = t->scr2.alloc(t->cfg.max_batch, Scratch::STREAM);
  if (e == hipSuccess && !t->stream_front)
    e = stream_beside(t->stream, reinterpret_cast<uint32_t*>(t->scr2.counters), &t->stream_front);
  if (e == hipSuccess && !t->ev_open) e = hipEventCreateWithFlags(&t->ev_open, hipEventDisableTiming);
  for (int k = 0; k < 2 && e == hipSuccess; ++k) {
    if (!t->ev_front[k]) e = hipEventCreateWithFlags(&t->ev_front[k], hipEventDisableTiming);
    if (e == hipSuccess && !t->ev_back[k])
      e = hipEventCreateWithFlags(&t->ev_back[k], hipEventDisableTiming);
  }
  if (e == hipSuccess) t->scr2_alloc = true;
  else {
    t->scr2.release();
    (void)hipGetLastError();  // or the next launch's check would find it
  }
  return e;
}

// Whether batches may overlap: the pipeline is there (stm_capture_graphs makes it at once), or the
// tree has seen enough batches for it to pay.  Making it takes 250 µs, and freeing it at the
// tree's end some 500 at a max_batch of 2^18 and more; a batch then gains 8 µs at 2^18 ops, 10 at
// 2^20, 15 at 2^22 (lookups on 2^22 keys).  Without the memory for it streams go on as before.
bool pipeline_ready(stm_tree* t) {
  if (t->scr2_alloc) return true;
  if (t->overlap_batches < OVERLAP_BATCHES || t->pipeline_failed) return false;
  t->pipeline_failed = make_pipeline(t) != hipSuccess;
  return t->scr2_alloc;
}

Scratch& slot_scratch(stm_tree* t, int k) { return k ? t->scr2 : t->scr; }

// Captures the launch sequence of size class c (on the first scratch set): advance (next descriptor
// of the window into the live descriptor), front half, back half.  Only classes up to
// GRAPH_MAX_OPS, and only when the caller asks (stm_capture_graphs): one call of the host replaces
// nine launches, but the kernels read their batch through the descriptor, which costs 6 µs of a
// 31 µs batch of 2^10 ops; above, the two halves on two streams are faster than any single graph
// (2^16 ops 69 against 87 µs, 2^18 ops 109 against 137).
int capture_class(stm_tree* t, int c) {
  if (t->graphs[c]) return STM_OK;
  Scratch& s = t->scr;
  hipStream_t st = t->stream;
  PipeIn in{nullptr, nullptr, nullptr, class_nmax(t, c), nullptr, nullptr, s.desc_live,
            false, nullptr, nullptr, 0, nullptr, s.acc};
  HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  k_advance<<<1, 64, 0, st>>>(s.desc_table, s.cursor, s.desc_live);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = enqueue_front(t, s, in, false, false, st);
  if (e == hipSuccess) e = enqueue_back(t, s, in, false);
  hipGraph_t g = nullptr;
  const hipError_t e2 = hipStreamEndCapture(st, &g);
  if (e == hipSuccess) e = e2;
  if (e == hipSuccess) e = hipGraphInstantiate(&t->graphs[c], g, nullptr, nullptr, 0);
  if (g) (void)hipGraphDestroy(g);
  if (e != hipSuccess) {
    t->graphs[c] = nullptr;
    return fail(STM_ERR_DEVICE, "graph capture of size class %d: %s", c, hipGetErrorString(e));
  }
  return STM_OK;
}

// Runs descs[at..] without a host round trip; ran = how many of them ran.  Fewer than all with
// STM_OK: the next one's small-batch sort overflowed a bucket, and it and the later ones ran empty.
//
// A batch runs in one of three ways, in order of size:
//   * a captured graph, where stm_capture_graphs made one for its class;
//   * both halves launched on the tree's stream: up to 2048 ops, whose front half is one short
//     kernel (per batch of 2^10 ops 31 µs, 41 with two streams), and while there is no second
//     scratch set and stream (pipeline_ready);
//   * the front half on stream_front once the back half of the scratch set's previous user is done,
//     the back half on the tree's stream once its front half is done (against one stream: 2^16 ops
//     69 / 79 µs, 2^18 109 / 129, 2^20 252 / 268, 2^22 657 / 669).
// Back halves run in batch order on one stream, so each sees the tree after the previous batch; the
// learned router retrains on that stream between them.  The first front half starts after
// whatever the caller had queued on the tree's stream: a copy into the batches' arrays, or out of
// the answers'.
int enqueue_descs(stm_tree* t, const std::vector<BatchDesc>& descs, const std::vector<uint8_t>& cls,
                  size_t at, size_t& ran, std::vector<BatchDesc>& table, StreamAcc& acc) {
  Scratch& s = t->scr;
  hipStream_t st = t->stream;
  ran = 0;
  int rc = maybe_retrain(t);  // learned routing: the router's buffers exist before capture
  if (rc) return rc;
  const bool exact_large = t->exact_left > 0, exact_small = t->front_hold > 0;
  auto replayed = [&](size_t i) {
    return descs[i].n <= GRAPH_MAX_OPS && t->graphs[cls[i]] && !exact_small;
  };
  bool normalized = false;  // batches whose sort may fall back for what the next ones hold too
  size_t replays = 0, large = 0;
  for (size_t i = at; i < descs.size(); ++i) {
    replays += replayed(i);
    large += descs[i].n >= OVERLAP_MIN_OPS;
    normalized |= descs[i].n > FRONT_MAX_OPS && !sample_sorted(descs[i].n);
  }
  t->overlap_batches += large;
  const bool overlap = large > 0 && pipeline_ready(t);
  hipStream_t sf = t->stream_front;
  bool used[2] = {false, false};  // ev_back[k] marks the end of the set's latest batch
  // Nothing to wait for on an idle stream: the wait of one stream for another costs 15 µs.
  if (overlap && hipStreamQuery(st) != hipSuccess) {
    (void)hipGetLastError();  // "not ready"
    HIP_TRY(hipEventRecord(t->ev_open, st));
    HIP_TRY(hipStreamWaitEvent(sf, t->ev_open, 0));
  }
  HIP_TRY(hipMemsetAsync(s.acc, 0, sizeof(StreamAcc), st));
  // The replayed batches' descriptors, window after window: a queued copy may still read those of
  // an earlier window.
  table.reserve(replays);
  int k = 0;  // the scratch set of the latest batch
  for (size_t w0 = at; w0 < descs.size(); w0 += DESC_TABLE) {
    const size_t w1 = std::min<size_t>(descs.size(), w0 + DESC_TABLE);
    const size_t first = table.size();
    for (size_t i = w0; i < w1; ++i)
      if (replayed(i)) table.push_back(descs[i]);
    if (table.size() > first) {
      HIP_TRY(hipMemcpyAsync(s.desc_table, table.data() + first,
                             (table.size() - first) * sizeof(BatchDesc), hipMemcpyHostToDevice, st));
      HIP_TRY(hipMemsetAsync(s.cursor, 0, sizeof(uint32_t), st));
    }
    for (size_t i = w0; i < w1; ++i) {
      const BatchDesc& d = descs[i];
      rc = maybe_retrain(t);
      if (rc) return rc;
      if (replayed(i)) {
        HIP_TRY(hipGraphLaunch(t->graphs[cls[i]], st));
        k = 0;
      } else {
        const PipeIn in{d.keys, d.vals, d.ops, d.n, d.out_vals, d.out_found, nullptr,
                        false, nullptr, nullptr, 0, nullptr, s.acc};
        const bool exact = d.n <= FRONT_MAX_OPS ? exact_small : exact_large && !sample_sorted(d.n);
        if (!overlap || d.n < OVERLAP_MIN_OPS) {
          HIP_TRY(enqueue_front(t, s, in, false, exact, st));
          HIP_TRY(enqueue_back(t, s, in, false));
          k = 0;
        } else {
          k ^= 1;
          Scratch& sk = slot_scratch(t, k);
          if (used[k]) HIP_TRY(hipStreamWaitEvent(sf, t->ev_back[k], 0));
          HIP_TRY(enqueue_front(t, sk, in, false, exact, sf));
          HIP_TRY(hipEventRecord(t->ev_front[k], sf));
          HIP_TRY(hipStreamWaitEvent(st, t->ev_front[k], 0));
          HIP_TRY(enqueue_back(t, sk, in, false));
        }
      }
      // A later batch's front half may take this scratch set on the other stream.
      if (overlap) {
        HIP_TRY(hipEventRecord(t->ev_back[k], st));
        used[k] = true;
      }
      t->st.batches += 1;
      t->st.ops += d.n;
      t->batches_since_train += 1;
    }
  }
  HIP_TRY(hipMemcpyAsync(&acc, s.acc, sizeof(acc), hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  ran = (size_t)acc.batches;
  if (acc.retries) {  // the failing batch and those after it did not run: taken out again
    for (size_t i = at + ran; i < descs.size(); ++i) t->st.ops -= descs[i].n;
    t->st.batches -= descs.size() - at - ran;
    t->batches_since_train -= (uint32_t)std::min<uint64_t>(t->batches_since_train, descs.size() - at - ran);
  }
  t->st.unique_ops += acc.unique;
  t->sort_fallbacks += acc.fallbacks;
  t->splits_since_train += acc.leaf_splits;
  if (acc.fallbacks && normalized) t->exact_left = EXACT_HOLD;
  else if (exact_large) t->exact_left -= (uint32_t)std::min<uint64_t>(t->exact_left, acc.batches);
  if (exact_small) t->front_hold -= (uint32_t)std::min<uint64_t>(t->front_hold, acc.batches);
  if (acc.sort_stalls)
    return fail(STM_ERR_DEVICE, "a batch sort gave up a grid-barrier wait (%llu later batches skipped)",
                acc.skipped);
  if (acc.bad)
    return fail(STM_ERR_INVALID, "a batch holds the reserved key 0xffffffffffffffff (%llu later batches skipped)",
                acc.skipped);
  rc = check_device_error(t);
  if (rc && acc.skipped) {
    char buf[64];
    snprintf(buf, sizeof(buf), " (%llu later batches skipped)", acc.skipped);
    g_last_error += buf;
  }
  return rc;
}

// enqueue_descs; after an error both streams are idle, as after success: what they still ran uses
// the scratch sets, the caller's arrays and the two copies' host memory here.
int run_descs(stm_tree* t, const std::vector<BatchDesc>& descs, const std::vector<uint8_t>& cls,
              size_t at, size_t& ran) {
  std::vector<BatchDesc> table;
  StreamAcc acc;
  const int rc = enqueue_descs(t, descs, cls, at, ran, table, acc);
  if (rc != STM_OK) {
    (void)hipStreamSynchronize(t->stream);
    if (t->stream_front) (void)hipStreamSynchronize(t->stream_front);
  }
  return rc;
}

int run_stream(stm_tree* t, const uint64_t* keys, const uint64_t* vals, const uint8_t* ops,
               const uint64_t* offsets, size_t nb, uint64_t* out_vals, uint8_t* out_found) {
  const uint64_t mb = t->cfg.max_batch;
  // Batches cut into chunks of at most max_batch ops, in order.
  std::vector<BatchDesc> descs;
  std::vector<uint8_t> cls;
  for (size_t b = 0; b < nb; ++b) {
    for (uint64_t off = offsets[b]; off < offsets[b + 1]; off += mb) {
      const uint32_t m = (uint32_t)std::min<uint64_t>(mb, offsets[b + 1] - off);
      descs.push_back(BatchDesc{keys + off, vals + off, ops + off, out_vals + off, out_found + off, m,
                                0, nullptr, nullptr, 0});
      cls.push_back((uint8_t)class_of(t, m));
    }
  }
  for (size_t at = 0; at < descs.size();) {
    size_t ran = 0;
    int rc = run_descs(t, descs, cls, at, ran);
    if (rc) return rc;
    at += ran;
    if (at >= descs.size()) break;
    // One batch's small-batch sort overflowed: it runs on its own with the exact sort (as do the
    // next EXACT_HOLD batches), then the stream goes on.
    t->front_hold = EXACT_HOLD + 1;
    t->sort_fallbacks += 1;
    const BatchDesc& d = descs[at++];
    rc = run_chunk(t, d.keys, d.vals, d.ops, d.n, d.out_vals, d.out_found);
    if (rc) return rc;
  }
  return STM_OK;
}

int validate_host_batch(const uint64_t* keys, const uint8_t* ops, size_t n, bool need_vals,
                        const uint64_t* vals) {
  bool any_insert = false;
  for (size_t i = 0; i < n; ++i) {
    if (keys[i] == STM_KEY_RESERVED)
      return fail(STM_ERR_INVALID, "op %zu uses the reserved key 0xffffffffffffffff", i);
    if (ops) {
      if (ops[i] > STM_OP_RANGE) return fail(STM_ERR_INVALID, "op %zu has op code %u", i, ops[i]);
      any_insert |= ops[i] == STM_OP_INSERT;
    }
  }
  if (need_vals && (any_insert || !ops) && !vals)
    return fail(STM_ERR_INVALID, "inserts need a value array");
  return STM_OK;
}

int run_device(stm_tree* t, const uint64_t* keys, const uint64_t* vals, const uint8_t* ops,
               size_t n, uint64_t* out_vals, uint8_t* out_found) {
  const uint64_t mb = t->cfg.max_batch;
  for (size_t off = 0; off < n; off += mb) {
    const uint32_t m = (uint32_t)std::min<uint64_t>(mb, n - off);
    int rc = run_chunk(t, keys + off, vals ? vals + off : nullptr, ops + off, m, out_vals + off,
                       out_found + off);
    if (rc) return rc;
  }
  return STM_OK;
}

// Bottom-up build of an empty tree from n device-resident pairs.
int build_from_device(stm_tree* t, const uint64_t* keys, const uint64_t* vals, size_t n) {
  hipStream_t st = t->stream;
  const uint32_t fill = t->cfg.leaf_fill;
  if (n > 0x7fffffffull) return fail(STM_ERR_INVALID, "bulk load of %zu keys exceeds 2^31-1", n);
  // The tree's own scratch when it is large enough, else one for this load.
  Scratch own;
  const bool fits = n <= t->scr.n;
  hipError_t e = fits ? hipSuccess : own.alloc(n, Scratch::LOAD);
  if (e != hipSuccess) {
    own.release();
    return fail(STM_ERR_NOMEM, "bulk-load scratch for %zu keys: %s", n, hipGetErrorString(e));
  }
  Scratch& tmp = fits ? t->scr : own;
  int rc = STM_OK;
  do {
    uint32_t U = 0;
    if (n > 0) {
      hipError_t r1 = radix_sort_pairs(keys, tmp.skeys_tmp, tmp.skeys, tmp.sidx_tmp, tmp.sidx,
                                       (uint32_t)n, 0, 64, tmp.hist, st);
      if (r1 != hipSuccess) { rc = fail(STM_ERR_DEVICE, "sort: %s", hipGetErrorString(r1)); break; }
      FoldArgs fa{};
      fa.skeys = tmp.skeys;
      fa.sidx = tmp.sidx;
      fa.vals = vals;
      fa.ops = nullptr;
      fa.n = (uint32_t)n;
      fa.ukey = tmp.ukey;
      fa.uval = tmp.uval;
      fa.uop = tmp.uop;
      fa.counters = tmp.counters;
      fa.tile_scratch = tmp.fold_tiles;
      fa.sort_stall = sort_stall_word(tmp.hist);
      r1 = fold_batch(fa, st);
      if (r1 != hipSuccess) { rc = fail(STM_ERR_DEVICE, "fold: %s", hipGetErrorString(r1)); break; }
      BatchCounters bc;
      if (hipMemcpyAsync(&bc, tmp.counters, sizeof(bc), hipMemcpyDeviceToHost, st) != hipSuccess ||
          hipStreamSynchronize(st) != hipSuccess) {
        rc = fail(STM_ERR_DEVICE, "bulk-load counters");
        break;
      }
      if (bc.sort_stall) { rc = fail(STM_ERR_DEVICE, "bulk-load sort: a grid-barrier wait gave up"); break; }
      if (bc.n_bad) { rc = fail(STM_ERR_INVALID, "bulk load holds the reserved key"); break; }
      U = bc.n_unique;
    }
    // Level sizes.
    std::vector<uint32_t> level_n;
    uint64_t L = U == 0 ? 1 : (U + fill - 1) / fill;
    level_n.push_back((uint32_t)L);
    while (level_n.back() > 1) level_n.push_back((level_n.back() + fill - 1) / fill);
    uint64_t total = 0;
    for (uint32_t c : level_n) total += c;
    if (total > t->capacity) {
      rc = fail(STM_ERR_NOMEM, "bulk load needs %llu nodes, pool holds %llu; raise max_keys",
                (unsigned long long)total, (unsigned long long)t->capacity);
      break;
    }
    // The levels' low fences ping-pong between the sort's key buffers, which the fold is done with.
    uint64_t *lows_a = tmp.skeys_tmp, *lows_b = tmp.skeys;
    hipError_t r2 = hipMemsetAsync(t->view.meta, 0, sizeof(NodeMeta) * t->capacity, st);
    if (r2 == hipSuccess)
      r2 = launch_build_leaves(t->view, tmp.ukey, tmp.uval, U, fill, (uint32_t)L, lows_a, st);
    uint32_t first_prev = 0, first_this = (uint32_t)L;
    uint64_t* lp = lows_a;
    uint64_t* lt = lows_b;
    for (size_t lv = 1; lv < level_n.size() && r2 == hipSuccess; ++lv) {
      r2 = launch_build_inner(t->view, lp, level_n[lv - 1], first_prev, fill, level_n[lv], first_this,
                              (uint32_t)lv, lt, st);
      first_prev = first_this;
      first_this += level_n[lv];
      std::swap(lp, lt);
    }
    if (r2 == hipSuccess) {
      TreeHeader h{};
      h.lock = 0;
      h.root = first_prev + level_n.back() - 1;
      if (level_n.size() == 1) h.root = 0;
      h.height = level_n.size();
      h.n_nodes = total;
      h.capacity = t->capacity;
      h.error = 0;
      h.n_keys = U;
      r2 = hipMemcpyAsync(t->view.hdr, &h, sizeof(h), hipMemcpyHostToDevice, st);
      if (r2 == hipSuccess)  // the key count restarts from the built tree
        r2 = hipMemsetAsync(t->view.stats + (size_t)ST_KEYS * STAT_STRIPES, 0,
                            sizeof(unsigned long long) * STAT_STRIPES, st);
      if (r2 == hipSuccess) r2 = hipStreamSynchronize(st);
      t->route_valid = false;  // the router describes the previous tree
      t->route_warm = false;
    }
    if (r2 != hipSuccess) rc = fail(STM_ERR_DEVICE, "bulk build: %s", hipGetErrorString(r2));
  } while (0);
  (void)hipStreamSynchronize(st);
  own.release();
  return rc;
}

// ------------------------------------------------------------------ batches without allocation
// stm_run_batch_device_noalloc keeps the scratch of its batch (sorted keys and positions, the
// sort's control words and histograms, fold tiles, per-group arrays, insert lists, counters)
// in this fixed device array instead of the tree's allocations.  Each GPU the library runs on
// holds its own copy until the process ends.  Host code never passes the array's name to a
// kernel or copy: it stands for a host-side shadow; the device address comes from
// hipGetSymbolAddress, once per device with that device current, and is kept per device.
constexpr size_t NOALLOC_BYTES = 8u << 20;
static __device__ __align__(256) uint8_t scratch[NOALLOC_BYTES];

struct NoAllocSlot {
  std::once_flag once;
  uint8_t* ptr = nullptr;  // device address of `scratch` on this device
  int rc = STM_OK;
  char err[192] = {};
};
constexpr int NOALLOC_DEVICES = 64;
NoAllocSlot g_noalloc[NOALLOC_DEVICES];

// Lays the batch scratch out in the device's copy of `scratch` (set up on the first call on
// the device: address lookup, then the sort's control words cleared).  Nothing is allocated.  The caller has made the tree's device current.
int noalloc_scratch(stm_tree* t, Scratch& s) {
  const int dev = t->cfg.device;
  if (dev < 0 || dev >= NOALLOC_DEVICES)
    return fail(STM_ERR_INVALID, "device %d outside the no-allocation table", dev);
  NoAllocSlot& d = g_noalloc[dev];
  std::call_once(d.once, [&] {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      d.rc = STM_ERR_DEVICE;
      snprintf(d.err, sizeof(d.err), "hipGetSymbolAddress: %s", hipGetErrorString(e));
      return;
    }
    Scratch probe;
    const size_t need = probe.carve(STM_NOALLOC_MAX_OPS, nullptr);
    if (need > NOALLOC_BYTES) {
      d.rc = STM_ERR_STATE;
      snprintf(d.err, sizeof(d.err), "layout of %zu bytes exceeds the %zu-byte array", need,
               NOALLOC_BYTES);
      return;
    }
    probe.carve(STM_NOALLOC_MAX_OPS, static_cast<uint8_t*>(p));
    e = sort_scratch_init(probe.hist);
    if (e != hipSuccess) {
      d.rc = STM_ERR_DEVICE;
      snprintf(d.err, sizeof(d.err), "sort control words: %s", hipGetErrorString(e));
      return;
    }
    d.ptr = static_cast<uint8_t*>(p);
  });
  if (d.rc != STM_OK) return fail(d.rc, "no-allocation scratch on device %d: %s", dev, d.err);
  s.carve(STM_NOALLOC_MAX_OPS, d.ptr);
  s.h_counters = t->scr.h_counters;  // pinned at stm_create
  return STM_OK;
}

}  // namespace

extern "C" {

const char* stm_last_error(void) { return g_last_error.c_str(); }

int stm_config_init(stm_config* cfg) {
  if (!cfg) return fail(STM_ERR_INVALID, "null config");
  std::memset(cfg, 0, sizeof(*cfg));
  cfg->fanout = 64;
  cfg->leaf_fill = 0;
  cfg->max_keys = 1ull << 24;
  cfg->max_batch = 1ull << 22;
  cfg->device = 0;
  cfg->lanes_per_op = 16;
  cfg->ops_per_group = 16;
  cfg->upsert_ops_per_wave = 512;
  cfg->max_attempts = 64;
  cfg->route = STM_ROUTE_DESCENT;
  cfg->timing = 0;
  cfg->retrain_every = 8;
  cfg->train_steps = 300;
  cfg->sort_tile_items = 16;
  cfg->use_graphs = 1;
  cfg->upsert_lanes = 0;  // automatic
  return STM_OK;
}

int stm_create(const stm_config* cfg_in, stm_tree** out) {
  if (!out) return fail(STM_ERR_INVALID, "null output handle");
  *out = nullptr;
  stm_config cfg;
  if (cfg_in) cfg = *cfg_in;
  else stm_config_init(&cfg);
  if (cfg.fanout != 32 && cfg.fanout != 64 && cfg.fanout != 128)
    return fail(STM_ERR_INVALID, "fanout %u not in {32, 64, 128}", cfg.fanout);
  if (cfg.leaf_fill == 0) cfg.leaf_fill = cfg.fanout - cfg.fanout / 4;
  if (cfg.leaf_fill < 2 || cfg.leaf_fill > cfg.fanout)
    return fail(STM_ERR_INVALID, "leaf_fill %u not in [2, fanout]", cfg.leaf_fill);
  if (cfg.max_batch == 0 || cfg.max_batch > (1ull << 30))
    return fail(STM_ERR_INVALID, "max_batch %llu not in [1, 2^30]", (unsigned long long)cfg.max_batch);
  if (cfg.max_keys == 0) return fail(STM_ERR_INVALID, "max_keys must be positive");
  const uint32_t lp = cfg.lanes_per_op;
  if (!(lp == 8 || lp == 16 || lp == 32 || lp == 64) || lp > cfg.fanout)
    return fail(STM_ERR_INVALID, "lanes_per_op %u not in {8,16,32,64} or above fanout", lp);
  if (cfg.ops_per_group == 0) cfg.ops_per_group = 16;
  if (cfg.upsert_ops_per_wave == 0) cfg.upsert_ops_per_wave = 512;
  if (cfg.sort_tile_items == 0) cfg.sort_tile_items = 16;
  if (cfg.sort_tile_items != 8 && cfg.sort_tile_items != 16)
    return fail(STM_ERR_INVALID, "sort_tile_items %u not in {8, 16}", cfg.sort_tile_items);
  // Kept for callers that set it; no kernel reads it.
  if (cfg.upsert_lanes == 0) cfg.upsert_lanes = cfg.fanout <= 64 ? 8u : 16u;
  if (!(cfg.upsert_lanes == 8 || cfg.upsert_lanes == 16 || cfg.upsert_lanes == 32) ||
      cfg.upsert_lanes > cfg.fanout)
    return fail(STM_ERR_INVALID, "upsert_lanes %u not in {8, 16, 32} or above fanout", cfg.upsert_lanes);
  if (cfg.max_attempts == 0) cfg.max_attempts = 64;
  if (cfg.retrain_every == 0) cfg.retrain_every = 8;
  if (cfg.train_steps > 100000) return fail(STM_ERR_INVALID, "train_steps above 100000");
  if (cfg.route > STM_ROUTE_INDEX) return fail(STM_ERR_INVALID, "route %u unknown", cfg.route);
  const uint64_t cap = capacity_for(cfg.max_keys, cfg.fanout);
  if (cap >= NODE_NONE) return fail(STM_ERR_INVALID, "max_keys too large for 32-bit node ids");

  stm_tree* t = new stm_tree();
  t->cfg = cfg;
  t->capacity = cap;
  int rc = set_device(t);
  if (rc) {
    delete t;
    return rc;
  }
  auto bail = [&](int code) {
    stm_destroy(t);
    return code;
  };
  if (hipStreamCreate(&t->stream) != hipSuccess) return bail(fail(STM_ERR_DEVICE, "hipStreamCreate"));
  const uint32_t F = cfg.fanout;
  hipError_t e = hipSuccess;
  auto pool_layout = [&](SlabCursor& cur) {
    t->view.keys = (uint64_t*)cur.take(sizeof(uint64_t) * cap * F);
    t->view.vals = (uint64_t*)cur.take(sizeof(uint64_t) * cap * F);
    t->view.meta = (NodeMeta*)cur.take(sizeof(NodeMeta) * cap);
    t->view.hdr = (TreeHeader*)cur.take(sizeof(TreeHeader));
    t->view.stats = (unsigned long long*)cur.take(sizeof(unsigned long long) * STATS_WORDS);
  };
  SlabCursor pool_size{nullptr};
  pool_layout(pool_size);
  if ((e = hipMalloc(&t->pool, pool_size.at)) == hipSuccess) {
    SlabCursor pool_place{(uint8_t*)t->pool};
    pool_layout(pool_place);
  } else
    return bail(fail(STM_ERR_NOMEM, "node pool of %llu nodes: %s", (unsigned long long)cap,
                     hipGetErrorString(e)));
  t->view.capacity = (uint32_t)cap;
  t->view.fanout = F;
  if ((e = t->scr.alloc(cfg.max_batch, Scratch::CALLS)) != hipSuccess)
    return bail(fail(STM_ERR_NOMEM, "batch scratch for %llu ops: %s",
                     (unsigned long long)cfg.max_batch, hipGetErrorString(e)));
  if (hipMemsetAsync(t->view.meta, 0, sizeof(NodeMeta) * cap, t->stream) != hipSuccess ||
      hipMemsetAsync(t->view.stats, 0, sizeof(unsigned long long) * STATS_WORDS, t->stream) != hipSuccess)
    return bail(fail(STM_ERR_DEVICE, "pool init"));
  // Phase events only time device work: without the system-scope fence a record is a
  // timestamp, not a cache write-back between two kernels (≈10 µs each at a phase boundary).
  for (int p = 0; p < STM_NUM_PHASES; ++p) {
    if (hipEventCreateWithFlags(&t->ev_a[p], hipEventDisableSystemFence) != hipSuccess ||
        hipEventCreateWithFlags(&t->ev_b[p], hipEventDisableSystemFence) != hipSuccess)
      return bail(fail(STM_ERR_DEVICE, "hipEventCreate"));
  }
  rc = init_empty(t);
  if (rc) return bail(rc);
  *out = t;
  return STM_OK;
}

int stm_destroy(stm_tree* t) {
  if (!t) return STM_OK;
  (void)hipSetDevice(t->cfg.device);
  if (t->stream) (void)hipStreamSynchronize(t->stream);
  if (t->stream_front) (void)hipStreamSynchronize(t->stream_front);
  drop_graphs(t);
  t->scr.release();
  if (t->scr2_alloc) t->scr2.release();
  if (t->ev_open) (void)hipEventDestroy(t->ev_open);
  for (int k = 0; k < 2; ++k) {
    if (t->ev_front[k]) (void)hipEventDestroy(t->ev_front[k]);
    if (t->ev_back[k]) (void)hipEventDestroy(t->ev_back[k]);
  }
  if (t->stream_front) (void)hipStreamDestroy(t->stream_front);
  if (t->pool) (void)hipFree(t->pool);
  for (int p = 0; p < STM_NUM_PHASES; ++p) {
    if (t->ev_a[p]) (void)hipEventDestroy(t->ev_a[p]);
    if (t->ev_b[p]) (void)hipEventDestroy(t->ev_b[p]);
  }
  free_router(t);
  if (t->stream) (void)hipStreamDestroy(t->stream);
  delete t;
  return STM_OK;
}

int stm_size(stm_tree* t, uint64_t* n_keys) {
  if (!t || !n_keys) return fail(STM_ERR_INVALID, "null argument");
  int rc = set_device(t);
  if (rc) return rc;
  TreeHeader h;
  rc = read_header(t, &h);
  if (rc) return rc;
  uint64_t c[ST_NUM];
  rc = read_counters(t, c);
  if (rc) return rc;
  *n_keys = h.n_keys + c[ST_KEYS];
  return STM_OK;
}

int stm_bulk_load_device(stm_tree* t, const uint64_t* d_keys, const uint64_t* d_vals, size_t n) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n && (!d_keys || !d_vals)) return fail(STM_ERR_INVALID, "null key or value array");
  int rc = set_device(t);
  if (rc) return rc;
  uint64_t have = 0;
  rc = stm_size(t, &have);
  if (rc) return rc;
  if (have == 0) return build_from_device(t, d_keys, d_vals, n);
  // Non-empty tree: a batch of inserts, outputs discarded into the staging buffers.
  const uint64_t mb = t->cfg.max_batch;
  HIP_TRY(hipMemsetAsync(t->scr.in_ops, STM_OP_INSERT, mb, t->stream));
  for (size_t off = 0; off < n; off += mb) {
    const uint32_t m = (uint32_t)std::min<uint64_t>(mb, n - off);
    rc = run_chunk(t, d_keys + off, d_vals + off, t->scr.in_ops, m, t->scr.out_vals, t->scr.out_found);
    if (rc) return rc;
  }
  return STM_OK;
}

int stm_bulk_load(stm_tree* t, const uint64_t* keys, const uint64_t* vals, size_t n) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n && (!keys || !vals)) return fail(STM_ERR_INVALID, "null key or value array");
  int rc = set_device(t);
  if (rc) return rc;
  rc = validate_host_batch(keys, nullptr, n, false, vals);
  if (rc) return rc;
  uint64_t *dk = nullptr, *dv = nullptr;
  if (dalloc(&dk, n) != hipSuccess || dalloc(&dv, n) != hipSuccess) {
    if (dk) (void)hipFree(dk);
    return fail(STM_ERR_NOMEM, "bulk-load input of %zu keys", n);
  }
  rc = STM_OK;
  if (n) {
    if (hipMemcpyAsync(dk, keys, n * 8, hipMemcpyHostToDevice, t->stream) != hipSuccess ||
        hipMemcpyAsync(dv, vals, n * 8, hipMemcpyHostToDevice, t->stream) != hipSuccess)
      rc = fail(STM_ERR_DEVICE, "bulk-load copy");
  }
  if (!rc) rc = stm_bulk_load_device(t, dk, dv, n);
  (void)hipStreamSynchronize(t->stream);
  (void)hipFree(dk);
  (void)hipFree(dv);
  return rc;
}

int stm_run_batch_device(stm_tree* t, const uint64_t* d_keys, const uint64_t* d_vals,
                         const uint8_t* d_ops, size_t n, uint64_t* d_out_vals, uint8_t* d_out_found) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n == 0) return STM_OK;
  if (!d_keys || !d_vals || !d_ops || !d_out_vals || !d_out_found)
    return fail(STM_ERR_INVALID, "null device array (device batches always carry values)");
  int rc = set_device(t);
  if (rc) return rc;
  return run_device(t, d_keys, d_vals, d_ops, n, d_out_vals, d_out_found);
}

int stm_run_batch_device_noalloc(stm_tree* t, const uint64_t* d_keys, const uint64_t* d_vals,
                                 const uint8_t* d_ops, size_t n, uint64_t* d_out_vals,
                                 uint8_t* d_out_found) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n == 0) return STM_OK;
  if (!d_keys || !d_vals || !d_ops || !d_out_vals || !d_out_found)
    return fail(STM_ERR_INVALID, "null device array (device batches always carry values)");
  if (n > STM_NOALLOC_MAX_OPS)
    return fail(STM_ERR_INVALID, "batch of %zu ops exceeds the %u ops the no-allocation scratch "
                "holds", n, (unsigned)STM_NOALLOC_MAX_OPS);
  int rc = set_device(t);
  if (rc) return rc;
  if (t->cfg.route != STM_ROUTE_DESCENT && !t->route_alloc)
    return fail(STM_ERR_STATE, "routing buffers do not exist yet: they are allocated by the first "
                "training (stm_retrain or one stm_run_batch_device call)");
  Scratch s;
  rc = noalloc_scratch(t, s);
  if (rc) return rc;
  return run_chunk(t, d_keys, d_vals, d_ops, (uint32_t)n, d_out_vals, d_out_found, nullptr, &s);
}

int stm_run_batches_device(stm_tree* t, const uint64_t* d_keys, const uint64_t* d_vals,
                           const uint8_t* d_ops, const uint64_t* offsets, size_t n_batches,
                           uint64_t* d_out_vals, uint8_t* d_out_found) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n_batches == 0) return STM_OK;
  if (!offsets) return fail(STM_ERR_INVALID, "null offsets");
  for (size_t b = 0; b < n_batches; ++b)
    if (offsets[b + 1] < offsets[b])
      return fail(STM_ERR_INVALID, "offsets decrease at batch %zu", b);
  if (offsets[n_batches] == offsets[0]) return STM_OK;
  if (!d_keys || !d_vals || !d_ops || !d_out_vals || !d_out_found)
    return fail(STM_ERR_INVALID, "null device array (device batches always carry values)");
  int rc = set_device(t);
  if (rc) return rc;
  // Flags in the place of op codes: a batch that has to be sorted again would find the ops of the
  // ones behind it gone.
  if (!t->cfg.use_graphs || overlaps(d_out_found + offsets[0], d_ops + offsets[0],
                                     offsets[n_batches] - offsets[0])) {
    for (size_t b = 0; b < n_batches; ++b) {
      const uint64_t o = offsets[b];
      rc = run_device(t, d_keys + o, d_vals + o, d_ops + o, offsets[b + 1] - o, d_out_vals + o,
                      d_out_found + o);
      if (rc) return rc;
    }
    return STM_OK;
  }
  return run_stream(t, d_keys, d_vals, d_ops, offsets, n_batches, d_out_vals, d_out_found);
}

int stm_run_batch_scan_device(stm_tree* t, const uint64_t* d_keys, const uint64_t* d_vals,
                              const uint8_t* d_ops, size_t n, uint64_t* d_out_vals,
                              uint8_t* d_out_found, uint64_t* d_scan_keys, uint64_t* d_scan_vals,
                              size_t scan_cap) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n == 0) return STM_OK;
  if (!d_keys || !d_vals || !d_ops || !d_out_vals || !d_out_found)
    return fail(STM_ERR_INVALID, "null device array (device batches always carry values)");
  if (scan_cap && (!d_scan_keys || !d_scan_vals)) return fail(STM_ERR_INVALID, "null scan area");
  int rc = set_device(t);
  if (rc) return rc;
  const uint64_t mb = t->cfg.max_batch;
  uint64_t base = 0;
  for (size_t off = 0; off < n; off += mb) {
    const uint32_t m = (uint32_t)std::min<uint64_t>(mb, n - off);
    ScanOut so{d_scan_keys ? d_scan_keys + base : nullptr, d_scan_vals ? d_scan_vals + base : nullptr,
               scan_cap - base, 0};
    rc = run_chunk(t, d_keys + off, d_vals + off, d_ops + off, m, d_out_vals + off,
                   d_out_found + off, &so);
    if (rc) return rc;
    base += std::min<uint64_t>(so.used, scan_cap - base);
  }
  return STM_OK;
}

int stm_run_batch_scan(stm_tree* t, const uint64_t* keys, const uint64_t* vals, const uint8_t* ops,
                       size_t n, uint64_t* out_vals, uint8_t* out_found, uint64_t* scan_keys,
                       uint64_t* scan_vals, size_t scan_cap) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n == 0) return STM_OK;
  if (!keys || !vals || !ops || !out_vals || !out_found) return fail(STM_ERR_INVALID, "null array");
  int rc = set_device(t);
  if (rc) return rc;
  rc = validate_host_batch(keys, ops, n, true, vals);
  if (rc) return rc;
  // Scan lengths: checked here, and each chunk's output area sized from them.
  const uint64_t mb = t->cfg.max_batch;
  std::vector<uint64_t> chunk_pairs;
  std::vector<ScanOp> scans;
  std::vector<size_t> chunk_scans{0};  // a chunk's scan ops begin here in `scans`
  uint64_t total = 0;
  for (size_t off = 0; off < n; off += mb) {
    const size_t m = (size_t)std::min<uint64_t>(mb, n - off);
    uint64_t c = 0;
    for (size_t i = off; i < off + m; ++i) {
      if (ops[i] != STM_OP_RANGE) continue;
      if (vals[i] < 1 || vals[i] > STM_SCAN_MAX_LEN)
        return fail(STM_ERR_INVALID, "scan op %zu has length %llu, not in [1, %u]", i,
                    (unsigned long long)vals[i], STM_SCAN_MAX_LEN);
      c += vals[i];
      scans.push_back(ScanOp{i, vals[i]});
    }
    chunk_pairs.push_back(c);
    chunk_scans.push_back(scans.size());
    total += c;
  }
  if (total > scan_cap)
    return fail(STM_ERR_INVALID, "scans need %llu pairs, the area holds %zu",
                (unsigned long long)total, scan_cap);
  if (total && (!scan_keys || !scan_vals)) return fail(STM_ERR_INVALID, "null scan area");
  const uint64_t most = *std::max_element(chunk_pairs.begin(), chunk_pairs.end());
  uint64_t *dsk = nullptr, *dsv = nullptr;
  if (dalloc(&dsk, most) != hipSuccess || dalloc(&dsv, most) != hipSuccess) {
    if (dsk) (void)hipFree(dsk);
    return fail(STM_ERR_NOMEM, "scan output area of %llu pairs", (unsigned long long)most);
  }
  Scratch& s = t->scr;
  std::unique_ptr<uint64_t[]> part;  // the area on the host, where scans left slots unwritten
  uint64_t base = 0;
  size_t ci = 0;
  for (size_t off = 0; off < n && rc == STM_OK; off += mb, ++ci) {
    const size_t m = (size_t)std::min<uint64_t>(mb, n - off);
    hipError_t e = hipMemcpyAsync(s.in_keys, keys + off, m * 8, hipMemcpyHostToDevice, t->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(s.in_vals, vals + off, m * 8, hipMemcpyHostToDevice, t->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(s.in_ops, ops + off, m, hipMemcpyHostToDevice, t->stream);
    if (e != hipSuccess) {
      rc = fail(STM_ERR_DEVICE, "batch copy: %s", hipGetErrorString(e));
      break;
    }
    ScanOut so{dsk, dsv, std::max<uint64_t>(most, 1), 0};
    rc = run_chunk(t, s.in_keys, s.in_vals, s.in_ops, (uint32_t)m, s.out_vals, s.out_found, &so);
    if (rc) break;
    const uint64_t c = chunk_pairs[ci];
    e = hipMemcpyAsync(out_vals + off, s.out_vals, m * 8, hipMemcpyDeviceToHost, t->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(out_found + off, s.out_found, m, hipMemcpyDeviceToHost, t->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    if (e == hipSuccess && c) {
      // The caller's slots past a scan's pairs stay as they are: straight into the caller's arrays
      // only when every slot was written.
      const ScanOp* sc = scans.data() + chunk_scans[ci];
      const size_t nsc = chunk_scans[ci + 1] - chunk_scans[ci];
      uint64_t wrote = 0;
      for (size_t q = 0; q < nsc; ++q) wrote += out_vals[sc[q].op];
      const bool whole = wrote == c;
      if (!whole && !part) part.reset(new (std::nothrow) uint64_t[most]);
      if (!whole && !part) {
        rc = fail(STM_ERR_NOMEM, "host copy of %llu scan pairs", (unsigned long long)most);
        break;
      }
      const uint64_t* from[] = {dsk, dsv};
      uint64_t* to[] = {scan_keys + base, scan_vals + base};
      for (int k = 0; k < 2 && e == hipSuccess; ++k) {
        e = hipMemcpyAsync(whole ? to[k] : part.get(), from[k], c * 8, hipMemcpyDeviceToHost, t->stream);
        if (e != hipSuccess || whole) continue;
        if ((e = hipStreamSynchronize(t->stream)) != hipSuccess) continue;
        written_pairs(sc, nsc, out_vals, [&](uint64_t at, uint64_t pairs) {
          std::memcpy(to[k] + at, part.get() + at, pairs * 8);
        });
      }
      if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
    }
    if (e != hipSuccess) rc = fail(STM_ERR_DEVICE, "result copy: %s", hipGetErrorString(e));
    base += c;
  }
  (void)hipStreamSynchronize(t->stream);
  (void)hipFree(dsk);
  (void)hipFree(dsv);
  return rc;
}

int stm_sort_pairs_device(int device, const uint64_t* d_keys, size_t n, uint64_t* d_keys_out,
                          uint32_t* d_idx_out) {
  if (n == 0) return STM_OK;
  if (!d_keys || !d_keys_out || !d_idx_out) return fail(STM_ERR_INVALID, "null device array");
  if (n > (1ull << 30)) return fail(STM_ERR_INVALID, "sort of %zu keys exceeds 2^30", n);
  HIP_TRY(hipSetDevice(device));
  uint64_t *ktmp = nullptr, *kin = nullptr;
  uint32_t *itmp = nullptr, *words = nullptr;
  void* slab = nullptr;
  int rc = STM_OK;
  // In place: the passes write the output before they have read the input for the last time.
  const bool apart = d_keys_out + n <= d_keys || d_keys + n <= d_keys_out;
  auto layout = [&](SlabCursor& cur) {
    ktmp = (uint64_t*)cur.take(n * 8);
    itmp = (uint32_t*)cur.take(n * 4);
    words = (uint32_t*)cur.take(sort_hist_words(n) * 4);
    if (!apart) kin = (uint64_t*)cur.take(n * 8);
  };
  SlabCursor size{nullptr};
  layout(size);
  if (hipMalloc(&slab, size.at) != hipSuccess) {
    slab = nullptr;
    rc = fail(STM_ERR_NOMEM, "sort scratch for %zu keys", n);
  } else {
    SlabCursor place{static_cast<uint8_t*>(slab)};
    layout(place);
    hipError_t e = sort_scratch_init(words);
    if (e == hipSuccess && kin)
      e = hipMemcpyAsync(kin, d_keys, n * 8, hipMemcpyDeviceToDevice, nullptr);
    if (e == hipSuccess)
      e = radix_sort_pairs(kin ? kin : d_keys, ktmp, d_keys_out, itmp, d_idx_out, (uint32_t)n, 0, 64, words,
                           nullptr);
    uint32_t stalled = 0;
    if (e == hipSuccess)
      e = hipMemcpy(&stalled, sort_stall_word(words), sizeof(stalled), hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = fail(STM_ERR_DEVICE, "sort: %s", hipGetErrorString(e));
    else if (stalled) rc = fail(STM_ERR_DEVICE, "sort: a bounded wait between workgroups gave up");
  }
  (void)hipDeviceSynchronize();
  if (slab) (void)hipFree(slab);
  return rc;
}

int stm_capture_graphs(stm_tree* t) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  int rc = set_device(t);
  if (rc) return rc;
  rc = maybe_retrain(t);  // learned routing: the router's buffers exist before capture
  if (rc) return rc;
  for (int c = 0; c < GRAPH_CLASSES && class_nmax(t, c) <= GRAPH_MAX_OPS; ++c) {
    rc = capture_class(t, c);
    if (rc) return rc;
    if (class_nmax(t, c) == t->cfg.max_batch) break;
  }
  const hipError_t e = make_pipeline(t);
  return e == hipSuccess ? STM_OK : fail(STM_ERR_NOMEM, "stream pipeline set-up: %s", hipGetErrorString(e));
}

int stm_run_batch(stm_tree* t, const uint64_t* keys, const uint64_t* vals, const uint8_t* ops,
                  size_t n, uint64_t* out_vals, uint8_t* out_found) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  if (n == 0) return STM_OK;
  if (!keys || !ops || !out_vals || !out_found) return fail(STM_ERR_INVALID, "null array");
  int rc = set_device(t);
  if (rc) return rc;
  rc = validate_host_batch(keys, ops, n, true, vals);
  if (rc) return rc;
  Scratch& s = t->scr;
  const uint64_t mb = t->cfg.max_batch;
  for (size_t off = 0; off < n; off += mb) {
    const size_t m = (size_t)std::min<uint64_t>(mb, n - off);
    HIP_TRY(hipMemcpyAsync(s.in_keys, keys + off, m * 8, hipMemcpyHostToDevice, t->stream));
    if (vals) HIP_TRY(hipMemcpyAsync(s.in_vals, vals + off, m * 8, hipMemcpyHostToDevice, t->stream));
    HIP_TRY(hipMemcpyAsync(s.in_ops, ops + off, m, hipMemcpyHostToDevice, t->stream));
    rc = run_chunk(t, s.in_keys, vals ? s.in_vals : nullptr, s.in_ops, (uint32_t)m, s.out_vals,
                   s.out_found);
    if (rc) return rc;
    HIP_TRY(hipMemcpyAsync(out_vals + off, s.out_vals, m * 8, hipMemcpyDeviceToHost, t->stream));
    HIP_TRY(hipMemcpyAsync(out_found + off, s.out_found, m, hipMemcpyDeviceToHost, t->stream));
    HIP_TRY(hipStreamSynchronize(t->stream));
  }
  return STM_OK;
}

int stm_dump(stm_tree* t, uint64_t* keys, uint64_t* vals, size_t cap, size_t* n) {
  if (!t || !n) return fail(STM_ERR_INVALID, "null argument");
  int rc = set_device(t);
  if (rc) return rc;
  TreeHeader h;
  rc = read_header(t, &h);
  if (rc) return rc;
  const uint32_t nn = (uint32_t)std::min<uint64_t>(h.n_nodes, t->capacity);
  hipStream_t st = t->stream;
  uint64_t *lows = nullptr, *slows = nullptr, *slows_tmp = nullptr, *offs = nullptr;
  uint32_t *ids = nullptr, *order = nullptr, *order_tmp = nullptr, *sorted_ids = nullptr,
           *counts = nullptr, *counter = nullptr, *hist = nullptr;
  uint64_t *ok = nullptr, *ov = nullptr;
  void *slab = nullptr, *out = nullptr;
  auto cleanup = [&]() {
    if (slab) (void)hipFree(slab);
    if (out) (void)hipFree(out);
  };
  auto err = [&](int code, const char* what) {
    (void)hipStreamSynchronize(st);
    cleanup();
    return fail(code, "dump: %s", what);
  };
  auto layout = [&](SlabCursor& cur) {
#define A_(p, c) p = static_cast<decltype(p)>(cur.take(sizeof(*p) * (size_t)(c)))
    A_(lows, nn); A_(slows, nn); A_(slows_tmp, nn); A_(ids, nn); A_(order, nn); A_(order_tmp, nn);
    A_(sorted_ids, nn); A_(counts, nn); A_(counter, 1); A_(offs, (size_t)nn + 1);
    A_(hist, sort_hist_words(nn));
#undef A_
  };
  SlabCursor size{nullptr};
  layout(size);
  if (hipMalloc(&slab, size.at) != hipSuccess) {
    slab = nullptr;
    return err(STM_ERR_NOMEM, "scratch");
  }
  SlabCursor place{static_cast<uint8_t*>(slab)};
  layout(place);
  if (sort_scratch_init(hist) != hipSuccess) return err(STM_ERR_DEVICE, "sort scratch");
  if (hipMemsetAsync(counter, 0, 4, st) != hipSuccess) return err(STM_ERR_DEVICE, "memset");
  if (launch_collect_leaves(t->view, nn, lows, ids, counter, st) != hipSuccess)
    return err(STM_ERR_DEVICE, "collect");
  uint32_t n_leaves = 0;
  if (hipMemcpyAsync(&n_leaves, counter, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return err(STM_ERR_DEVICE, "leaf count");
  if (radix_sort_pairs(lows, slows_tmp, slows, order_tmp, order, n_leaves, 0, 64, hist, st) != hipSuccess ||
      launch_leaf_counts(t->view, order, ids, n_leaves, sorted_ids, counts, st) != hipSuccess)
    return err(STM_ERR_DEVICE, "leaf order");
  uint32_t stalled = 0;
  if (hipMemcpyAsync(&stalled, sort_stall_word(hist), 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return err(STM_ERR_DEVICE, "leaf order");
  if (stalled) return err(STM_ERR_DEVICE, "leaf order: a sort grid-barrier wait gave up");
  std::vector<uint32_t> hc(n_leaves);
  if (n_leaves && (hipMemcpyAsync(hc.data(), counts, 4ull * n_leaves, hipMemcpyDeviceToHost, st) != hipSuccess ||
                   hipStreamSynchronize(st) != hipSuccess))
    return err(STM_ERR_DEVICE, "counts");
  std::vector<uint64_t> ho(n_leaves + 1, 0);
  for (uint32_t r = 0; r < n_leaves; ++r) ho[r + 1] = ho[r] + hc[r];
  const uint64_t total = ho[n_leaves];
  *n = total;
  if (!keys || !vals || cap < total) {
    (void)hipStreamSynchronize(st);
    cleanup();
    if (!keys && !vals && cap == 0) return STM_OK;  // size query
    return fail(STM_ERR_INVALID, "dump needs room for %llu pairs, got %zu", (unsigned long long)total, cap);
  }
  if (total && hipMalloc(&out, total * 16) != hipSuccess) {
    out = nullptr;
    return err(STM_ERR_NOMEM, "output");
  }
  ok = static_cast<uint64_t*>(out);
  ov = ok + total;
  if (hipMemcpyAsync(offs, ho.data(), 8ull * (n_leaves + 1), hipMemcpyHostToDevice, st) != hipSuccess ||
      launch_dump_copy(t->view, sorted_ids, offs, n_leaves, ok, ov, st) != hipSuccess)
    return err(STM_ERR_DEVICE, "copy");
  if (total && (hipMemcpyAsync(keys, ok, total * 8, hipMemcpyDeviceToHost, st) != hipSuccess ||
                hipMemcpyAsync(vals, ov, total * 8, hipMemcpyDeviceToHost, st) != hipSuccess))
    return err(STM_ERR_DEVICE, "download");
  if (hipStreamSynchronize(st) != hipSuccess) return err(STM_ERR_DEVICE, "sync");
  cleanup();
  return STM_OK;
}

int stm_check(stm_tree* t, uint64_t* bad) {
  if (!t || !bad) return fail(STM_ERR_INVALID, "null argument");
  int rc = set_device(t);
  if (rc) return rc;
  TreeHeader h;
  rc = read_header(t, &h);
  if (rc) return rc;
  unsigned long long* d = nullptr;
  HIP_TRY(dalloc(&d, 1));
  unsigned long long v = 0;
  hipError_t e = hipMemsetAsync(d, 0, 8, t->stream);
  const uint32_t nn = (uint32_t)std::min<uint64_t>(h.n_nodes, t->capacity);
  if (e == hipSuccess) e = launch_check(t->view, nn, d, t->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(&v, d, 8, hipMemcpyDeviceToHost, t->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
  (void)hipFree(d);
  if (e != hipSuccess) return fail(STM_ERR_DEVICE, "check: %s", hipGetErrorString(e));
  // Root and height must describe a node of the right level.
  NodeMeta rm;
  HIP_TRY(hipMemcpy(&rm, t->view.meta + h.root, sizeof(rm), hipMemcpyDeviceToHost));
  if (meta_level(rm.info) + 1 != h.height || rm.low != 0 || rm.high != KEY_EMPTY) v++;
  *bad = v;
  return STM_OK;
}

int stm_get_stats(stm_tree* t, stm_stats* out) {
  if (!t || !out) return fail(STM_ERR_INVALID, "null argument");
  int rc = set_device(t);
  if (rc) return rc;
  TreeHeader h;
  rc = read_header(t, &h);
  if (rc) return rc;
  uint64_t c[ST_NUM];
  rc = read_counters(t, c);
  if (rc) return rc;
  *out = t->st;
  out->n_keys = h.n_keys + c[ST_KEYS];
  out->n_nodes = std::min<uint64_t>(h.n_nodes, t->capacity);
  out->capacity_nodes = t->capacity;
  out->height = h.height;
  out->upserts = c[ST_UPSERTS];
  out->commits = c[ST_COMMITS];
  out->aborts = c[ST_ABORTS];
  out->leaf_splits = c[ST_LEAF_SPLITS];
  out->inner_splits = c[ST_INNER_SPLITS];
  out->root_splits = c[ST_ROOT_SPLITS];
  out->deferred = c[ST_DEFERRED];
  out->route_hits = c[ST_ROUTE_HITS];
  out->route_misses = c[ST_ROUTE_MISSES];
  out->node_reads = c[ST_NODE_READS];
  out->leaf_steps = c[ST_LEAF_STEPS];
  out->sort_fallbacks = t->sort_fallbacks;
  return STM_OK;
}

int stm_retrain(stm_tree* t, uint32_t train_steps) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  int rc = set_device(t);
  if (rc) return rc;
  rc = train_router(t, train_steps, false);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(t->stream));
  phase_collect(t);
  return STM_OK;
}

int stm_route_info(stm_tree* t, uint64_t* n_leaves, uint64_t* window_hits, uint64_t* window_misses) {
  if (!t || !n_leaves || !window_hits || !window_misses) return fail(STM_ERR_INVALID, "null argument");
  if (!t->route_valid) return fail(STM_ERR_STATE, "no router has been trained (stm_retrain)");
  int rc = set_device(t);
  if (rc) return rc;
  uint64_t* d = nullptr;
  HIP_TRY(dalloc(&d, 2));
  uint64_t hm[2] = {0, 0};
  hipError_t e = hipMemsetAsync(d, 0, 16, t->stream);
  if (e == hipSuccess) e = route_evaluate(t->route, d, (uint32_t)t->capacity, t->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(hm, d, 16, hipMemcpyDeviceToHost, t->stream);
  RouteHeader rh{};
  if (e == hipSuccess) e = hipMemcpyAsync(&rh, t->route.hdr, sizeof(rh), hipMemcpyDeviceToHost, t->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(t->stream);
  (void)hipFree(d);
  if (e != hipSuccess) return fail(STM_ERR_DEVICE, "route info: %s", hipGetErrorString(e));
  *n_leaves = rh.L;
  *window_hits = hm[0];
  *window_misses = hm[1];
  return STM_OK;
}

int stm_route_directory(stm_tree* t, uint64_t* fences, uint32_t* leaf_ids, uint64_t max,
                        uint64_t* n_leaves) {
  if (!t || !n_leaves || (!fences != !leaf_ids)) return fail(STM_ERR_INVALID, "null argument");
  if (!t->route_valid) return fail(STM_ERR_STATE, "no router has been trained (stm_retrain)");
  int rc = set_device(t);
  if (rc) return rc;
  RouteHeader rh{};
  HIP_TRY(hipMemcpyAsync(&rh, t->route.hdr, sizeof(rh), hipMemcpyDeviceToHost, t->stream));
  HIP_TRY(hipStreamSynchronize(t->stream));
  *n_leaves = rh.L;
  if (!fences) return STM_OK;  // size query
  if (rh.L > max) return fail(STM_ERR_INVALID, "directory holds %u leaves, room for %llu", rh.L,
                              (unsigned long long)max);
  if (rh.L) {
    HIP_TRY(hipMemcpyAsync(fences, t->route.fences, sizeof(uint64_t) * rh.L, hipMemcpyDeviceToHost,
                           t->stream));
    HIP_TRY(hipMemcpyAsync(leaf_ids, t->route.lids, sizeof(uint32_t) * rh.L, hipMemcpyDeviceToHost,
                           t->stream));
    HIP_TRY(hipStreamSynchronize(t->stream));
  }
  return STM_OK;
}

int stm_mlp_gradients(const float* x, const float* tg, size_t n, const float* params49,
                      float* grad49, float* loss) {
  if (!params49 || !grad49 || !loss || (n && (!x || !tg))) return fail(STM_ERR_INVALID, "null argument");
  if (n > (1u << 24)) return fail(STM_ERR_INVALID, "at most 2^24 pairs");
  float *dx = nullptr, *dt = nullptr, *dp = nullptr, *dg = nullptr, *dl = nullptr;
  int rc = STM_OK;
  if (dalloc(&dx, n) || dalloc(&dt, n) || dalloc(&dp, MLP_PARAMS) || dalloc(&dg, MLP_PARAMS) ||
      dalloc(&dl, 1)) {
    rc = fail(STM_ERR_NOMEM, "gradient buffers");
  } else {
    hipError_t e = hipSuccess;
    if (n) e = hipMemcpy(dx, x, n * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess && n) e = hipMemcpy(dt, tg, n * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dp, params49, MLP_PARAMS * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = mlp_grad(dx, dt, (uint32_t)n, dp, dg, dl, nullptr);
    if (e == hipSuccess) e = hipMemcpy(grad49, dg, MLP_PARAMS * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(loss, dl, 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) rc = fail(STM_ERR_DEVICE, "mlp gradients: %s", hipGetErrorString(e));
  }
  void* ps[] = {dx, dt, dp, dg, dl};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  return rc;
}

int stm_reset_stats(stm_tree* t) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  int rc = set_device(t);
  if (rc) return rc;
  t->st = stm_stats{};
  t->sort_fallbacks = 0;
  HIP_TRY(hipMemsetAsync(t->view.stats, 0, sizeof(unsigned long long) * STATS_RESET_WORDS, t->stream));
  HIP_TRY(hipStreamSynchronize(t->stream));
  return STM_OK;
}

int stm_get_stream(stm_tree* t, void** stream) {
  if (!t || !stream) return fail(STM_ERR_INVALID, "null argument");
  *stream = (void*)t->stream;
  return STM_OK;
}

int stm_device_alloc(int device, size_t bytes, void** ptr) {
  if (!ptr) return fail(STM_ERR_INVALID, "null argument");
  *ptr = nullptr;
  HIP_TRY(hipSetDevice(device));
  HIP_TRY(hipMalloc(ptr, bytes ? bytes : 1));
  return STM_OK;
}

int stm_device_free(void* ptr) {
  if (ptr) HIP_TRY(hipFree(ptr));
  return STM_OK;
}

int stm_memcpy_h2d(void* dst, const void* src, size_t bytes) {
  if (!bytes) return STM_OK;
  if (!dst || !src) return fail(STM_ERR_INVALID, "null argument");
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
  return STM_OK;
}

int stm_memcpy_d2h(void* dst, const void* src, size_t bytes) {
  if (!bytes) return STM_OK;
  if (!dst || !src) return fail(STM_ERR_INVALID, "null argument");
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return STM_OK;
}

int stm_device_copy(void* dst, const void* src, size_t bytes) {
  if (!bytes) return STM_OK;
  if (!dst || !src) return fail(STM_ERR_INVALID, "null argument");
  if ((bytes & 15) || ((uintptr_t)dst & 15) || ((uintptr_t)src & 15))
    return fail(STM_ERR_INVALID, "device copy needs 16-byte aligned pointers and size");
  const uint64_t n16 = bytes / 16;
  const uint32_t blocks = (uint32_t)std::min<uint64_t>((n16 + 255) / 256, COPY_MAX_BLOCKS);
  k_copy16<<<blocks, 256, 0, nullptr>>>((uint4*)dst, (const uint4*)src, n16);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipDeviceSynchronize());
  return STM_OK;
}

int stm_sync(stm_tree* t) {
  if (!t) return fail(STM_ERR_INVALID, "null tree");
  HIP_TRY(hipStreamSynchronize(t->stream));
  return STM_OK;
}

}  // extern "C"
