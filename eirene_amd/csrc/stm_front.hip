// stm_front.hip — front half of a batch of at most FRONT_MAX_OPS ops: stable sort by key and
// per-key fold (the same results as stm_sort.hip and stm_fold.hip, which serve larger batches).
//
// A batch of this size is bound by latency, not by bytes: each launch costs 2-4 µs and each
// dependent round trip to memory about 1 µs, whatever they move.  So the front half is built for
// few launches and few round trips, and sorts in LDS (stm_binsort.hpp), where the exact key and
// the input position are one 96-bit value: no normalization, no second pass over near-equal keys,
// and equal keys need no special care.
//
//   up to FRONT_SMALL ops, one workgroup:
//     k_front_small   sort in LDS, fold, outputs
//   above, three launches:
//     k_front_split   every workgroup sorts the same sample of the batch, takes every
//                     OVERSAMPLE-th as a splitter and orders its own tile by bucket
//     k_front_bucket  one workgroup per bucket collects its pieces from the tiles and sorts them
//     k_front_fold    one workgroup per bucket: the bucket's place among the groups from the
//                     other buckets' summaries, then the fold's outputs
// Sorts outside of batches (front_sort: a tree's leaves, loads, stm_sort_pairs_device) take the same
// kernels without the fold, k_front_keys in the place of k_front_small.
//
// The radix form this replaces took ten or eleven launches: k_range, the digit histograms and
// their scan, two or three single-sweep passes, the bucket fix-up, the exact-sort check and three
// fold kernels.  Kernel times, replaced / now: 1000 ops 52 / 7.0 µs, 40001 ops 86 / 26 µs, 131075 ops
// 101 / 38 µs; most of what is left is three round trips to memory per kernel and the barriers
// between the steps of a workgroup's sort.
//
// Buckets are cut between samples of (key, position), so a hot key's ops are shared by as many
// buckets as they fill.  With OVERSAMPLE samples per bucket drawn at hashed positions, one per
// equal stretch of the input, a bucket holds more than BUCKET_CAP elements (at least four times
// the mean) about once in 10^5 batches of the largest size if the input is not built to
// mislead the sample.  The batch then runs empty (sort_retry) and the caller sorts it again with
// the exact radix passes.
#include <algorithm>

#include "stm_binsort.hpp"
#include "stm_common.hpp"
#include "stm_fold.hpp"
#include "stm_internal.hpp"

namespace stm {

constexpr uint32_t FRONT_SMALL = 2 * FT;
constexpr uint32_t OVERSAMPLE = 8;
constexpr uint32_t BUCKETS_MAX = 256;
constexpr uint32_t BUCKET_CAP = 4 * FT;
constexpr uint32_t TILES_MAX = FRONT_MAX_OPS / (2 * FT);

// Front scratch (u32 words): the retry flag, then each bucket's first sorted position and its
// summary, then per tile the first element of every bucket within the tile.
struct BucketSum {
  uint32_t start;  // sorted position of the bucket's first element
  Acc acc;         // its elements, the first one not counted as a head
};
static_assert(sizeof(BucketSum) == 20, "five words");
constexpr uint32_t FRONT_RETRY = 0;
constexpr uint32_t FRONT_SUMS = 64;
constexpr uint32_t FRONT_OFFS = FRONT_SUMS + 5 * BUCKETS_MAX;
constexpr uint32_t FRONT_WORDS = FRONT_OFFS + TILES_MAX * (BUCKETS_MAX + 1);
size_t front_scratch_words() { return FRONT_WORDS; }

// ------------------------------------------------------------------ fold of sorted elements
// One sorted element as the fold sees it (a thread's own).
struct FoldElem {
  bool valid, ins, end;  // in the batch; an INSERT; the last element of its group
  int32_t i, head, lb;   // sorted position, its group's head, the latest earlier insert of the key (-1)
  uint32_t g;            // group index
  uint32_t e;            // the group's place in the insert list (a group with an INSERT)
  uint64_t key;
  uint32_t pos, lb_pos;  // input positions of the element and of lb
  uint64_t va, vb;       // lb's value, the element's own (loaded where needed)
};

STM_DEV void fold_gather(const FoldArgs& a, FoldElem& x) {
  const bool real = x.key != KEY_EMPTY;
  const bool need_a = x.valid && x.lb >= 0 && (a.out_vals || (x.end && !x.ins && real));
  const bool need_b = x.valid && x.end && x.ins && real;
  x.va = need_a ? a.vals[x.lb_pos] : 0ull;
  x.vb = need_b ? a.vals[x.pos] : 0ull;
}

// Writes the element's outputs.  Ops with the reserved key are added to bad, and answered as absent.
STM_DEV void fold_store(const FoldArgs& a, const FoldElem& x, uint32_t* bad) {
  if (!x.valid) return;
  if (a.lastins) a.lastins[x.i] = x.ins ? x.i : x.lb;
  if (x.lb >= 0) {
    a.out_vals[x.pos] = x.va;  // out_found stays 1
  }
  if (x.key == KEY_EMPTY) {
    a.out_vals[x.pos] = 0;
    a.out_found[x.pos] = 0;
  }
  if (x.ins && x.lb < 0) a.npend[x.g] = (uint32_t)(x.i - x.head + 1);
  if (!x.end) return;
  a.ukey[x.g] = x.key;
  a.gstart[x.g] = (uint32_t)x.head;
  const int32_t last_in = x.ins ? x.i : x.lb;  // the group's last insert
  if (x.key == KEY_EMPTY) {
    a.uop[x.g] = UOP_SKIP;
    atomicAdd(bad, (uint32_t)(x.i - x.head + 1));
  } else if (last_in >= 0) {
    a.uop[x.g] = OP_INSERT;
    a.uval[x.g] = x.ins ? x.vb : x.va;
    a.ilist[x.e] = x.g;
  } else {
    a.uop[x.g] = OP_GET;
    a.npend[x.g] = (uint32_t)(x.i - x.head + 1);
  }
}

// Head, insert, group and list fields of this thread's element from the state before its
// wavefront's 64 elements, which start at sorted position rb and have heads hm and INSERTs im.
STM_DEV void fold_place(FoldElem& x, uint64_t hm, uint64_t im, uint32_t rb, const Acc& before) {
  const uint64_t lt = lanemask_lt();
  const uint64_t le = lt | (1ull << lane_id());
  x.head = last_set(hm & le, rb, before.head);
  const int32_t ins_before = last_set(im & lt, rb, before.ins);
  x.lb = ins_before >= x.head ? ins_before : -1;
  x.g = before.c + (uint32_t)__popcll(hm & le) - 1;
  const uint64_t fm = first_inserts(hm, im, acc_open_insert(before));
  x.e = (before.m & ~ACC_LEAD) + (uint32_t)__popcll(fm & le) - 1;
}

// Combination, in lane order, of the 64 lanes' states (complete in lane 0).
STM_DEV Acc wave_combine(Acc v) {
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const Acc o{(uint32_t)__shfl_down((int)v.c, off, WAVE), __shfl_down(v.head, off, WAVE),
                __shfl_down(v.ins, off, WAVE), (uint32_t)__shfl_down((int)v.m, off, WAVE)};
    if (lane_id() + off < WAVE) v = acc_combine(v, o);
  }
  return v;
}

// Up to FT * E keys without op codes, sorted by one workgroup.
template <int E>
__global__ __launch_bounds__(FT) void k_front_keys(FrontSort fs) {
  constexpr uint32_t N = FT * E;
  __shared__ uint64_t s_k[N];
  __shared__ uint32_t s_p[N];
  __shared__ BinShared s_bin;
  const uint32_t n = min(fs.n, N);
  const uint32_t tid = threadIdx.x;
  uint64_t k[E];
  uint32_t p[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    k[r] = i < n ? gload(fs.keys + i) : KEY_EMPTY;
    p[r] = i < n ? i : ~0u;
  }
  if (tid == 0) {
    *fs.need = 0;
    *fs.stall = 0;
  }
  bin_sort_open<FT>(s_bin);
  __syncthreads();
  bin_sort<FT, E>(n, k, p, s_k, s_p, s_bin);
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    if (i < n) {
      fs.keys_out[i] = s_k[i];
      fs.idx_out[i] = s_p[i];
    }
  }
}

struct FrontIn {
  const uint64_t* keys;
  const uint8_t* ops;
  uint32_t n;
};
STM_DEV FrontIn front_in(const FrontArgs& a) {
  const BatchDesc* d = a.fold.desc;
  return d ? FrontIn{d->keys, d->ops, d->n} : FrontIn{a.keys, a.ops, a.fold.n};
}

STM_DEV void reset_counters(BatchCounters* c, uint32_t groups, uint32_t upserts, uint32_t bad) {
  c->n_unique = groups;
  c->n_upserts = upserts;
  c->n_deferred = 0;
  c->queue_head = 0;
  c->n_bad = bad;
  c->n_fanout = 0;
  c->sort_stall = 0;
  c->sort_fallback = 0;
  c->sort_retry = 0;
  c->leaf_splits = 0;
}

// The whole front half of a batch of at most FT * E ops, in one workgroup.
template <int E>
__global__ __launch_bounds__(FT) void k_front_small(FrontArgs fa) {
  constexpr uint32_t N = FT * E;
  constexpr int CHUNKS = FW * E;  // 64-element chunks of the sorted batch
  __shared__ uint64_t s_k[N];
  __shared__ uint32_t s_p[N];
  __shared__ Acc s_acc[CHUNKS];
  __shared__ BinShared s_bin;
  __shared__ uint32_t s_bad;
  const FrontIn in = front_in(fa);
  FoldArgs a = fa.fold;
  fold_resolve(a);
  const uint32_t n = min(in.n, N);
  const uint32_t tid = threadIdx.x;
  const uint32_t wave = tid / WAVE;
  uint64_t k[E];
  uint32_t p[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    const bool v = i < n;
    const uint64_t kk = v ? gload(in.keys + i) : KEY_EMPTY;
    const uint32_t op = v ? gload(in.ops + i) : 0u;
    k[r] = kk;
    p[r] = v ? tie_of(i, op) : ~0u;
    if (v) a.out_found[i] = 1;  // the answers' default
  }
  bin_sort_open<FT>(s_bin);
  if (tid == 0) s_bad = 0;
  __syncthreads();
  bin_sort<FT, E>(n, k, p, s_k, s_p, s_bin);
  FoldElem x[E];
  uint64_t hm[E], im[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    x[r].valid = i < n;
    x[r].i = (int32_t)i;
    x[r].key = s_k[i];
    const uint32_t tie = s_p[i];
    x[r].pos = tie >> 2;
    x[r].ins = x[r].valid && (tie & 3u) == OP_INSERT && x[r].key != KEY_EMPTY;
    hm[r] = ballot(x[r].valid && (i == 0 || s_k[i > 0 ? i - 1 : 0] != x[r].key));
    im[r] = ballot(x[r].ins);
    x[r].end = x[r].valid && (i + 1 >= n || s_k[min(i + 1, N - 1)] != x[r].key);
    const uint32_t rb = (uint32_t)r * FT + wave * WAVE;
    if (lane_id() == 0) s_acc[rb / WAVE] = acc_round(acc_identity(), hm[r], im[r], rb);
    if (x[r].valid) const_cast<uint32_t*>(a.sidx)[i] = payload_of(tie);
  }
  __syncthreads();
  Acc run = acc_identity();
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const Acc t = s_acc[c];
#pragma unroll
    for (int r = 0; r < E; ++r)
      if ((uint32_t)c == (uint32_t)r * FW + wave)
        fold_place(x[r], hm[r], im[r], (uint32_t)c * WAVE, run);
    run = acc_combine(run, t);
  }
#pragma unroll
  for (int r = 0; r < E; ++r) {
    x[r].lb_pos = x[r].valid && x[r].lb >= 0 ? s_p[x[r].lb] >> 2 : 0u;
    fold_gather(a, x[r]);
  }
#pragma unroll
  for (int r = 0; r < E; ++r) fold_store(a, x[r], &s_bad);
  __syncthreads();
  if (tid == 0) reset_counters(a.counters, run.c, run.m & ~ACC_LEAD, s_bad);
}

// ------------------------------------------------------------------ split
// Tile blockIdx.x of FT * E elements, ordered by bucket into tmp (the order within a bucket does
// not matter: the bucket sort compares positions too).  Every workgroup sorts the same S samples
// itself, which costs less than a launch for it and the round trip that reads the result.
// BATCH: with op codes, found flags to set to their default and counters to reset.
template <int E, int S, bool BATCH>
__global__ __launch_bounds__(FT) void k_front_split(FrontArgs fa) {
  constexpr uint32_t TILE = FT * E;
  constexpr int B = S / (int)OVERSAMPLE;
  constexpr int SE = S > FT ? S / FT : 1;  // samples per thread
  constexpr int SN = FT * SE;
  __shared__ uint64_t s_k[SN];
  __shared__ uint32_t s_p[SN];
  __shared__ BinShared s_bin;
  __shared__ uint32_t s_cnt[B], s_off[B + 1];
  __shared__ uint32_t s_w[FW];
  const FrontIn in = front_in(fa);
  const uint32_t n = in.n;
  const uint32_t tid = threadIdx.x;
  uint8_t* found = fa.fold.desc ? fa.fold.desc->out_found : fa.fold.out_found;
  if (blockIdx.x == 0 && tid == 0) {
    if constexpr (BATCH) {
      reset_counters(fa.fold.counters, 0, 0, 0);
    } else {
      *fa.stall = 0;
      *fa.barrier = 0;
    }
    *fa.retry = 0;
  }
  if ((uint64_t)blockIdx.x * TILE >= n) return;
  const uint32_t tile0 = blockIdx.x * TILE;
  const uint32_t tile_n = min(TILE, n - tile0);
  // The tile's own elements travel while the samples are sorted.
  uint64_t ek[E];
  uint32_t ep[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t le = min((uint32_t)r * FT + tid, tile_n - 1);
    ek[r] = gload(in.keys + tile0 + le);
    ep[r] = BATCH ? gload(in.ops + tile0 + le) : 0u;
  }
  uint64_t sk[SE];
  uint32_t sp[SE];
#pragma unroll
  for (int r = 0; r < SE; ++r) {
    const uint32_t j = (uint32_t)r * FT + tid;
    sk[r] = KEY_EMPTY;
    sp[r] = ~0u;
    if (j < (uint32_t)S) {
      // One sample from each of S equal stretches of the input, at a hashed place.
      const uint32_t lo = (uint32_t)((uint64_t)j * n / S);
      const uint32_t hi = (uint32_t)((uint64_t)(j + 1) * n / S);
      const uint32_t at = min(lo + (uint32_t)(((uint64_t)hash32(j) * (hi - lo)) >> 32), n - 1);
      sk[r] = gload(in.keys + at);
      sp[r] = at << 2;
    }
  }
  if (tid < (uint32_t)B) s_cnt[tid] = 0;
  if constexpr (S < FT) {  // few enough for the comparison sort, and indifferent to crowded keys
    block_sort<S, 1>(sk, sp, s_k, s_p);
    __syncthreads();
    if (tid < (uint32_t)S) {
      s_k[tid] = sk[0];
      s_p[tid] = sp[0];
    }
    __syncthreads();
  } else {
    bin_sort_open<FT>(s_bin);
    __syncthreads();
    bin_sort<FT, SE>(S, sk, sp, s_k, s_p, s_bin);
  }
  // Bucket: the splitters 1 .. B - 1 not above the element.
  uint32_t bkt[E], rank[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t le = (uint32_t)r * FT + tid;
    ep[r] = tie_of(tile0 + le, ep[r]);
    uint32_t lo = 0;
#pragma unroll
    for (int step = B / 2; step > 0; step >>= 1) {
      const uint32_t q = lo + (uint32_t)step;
      if (!elem_less(ek[r], ep[r], s_k[q * OVERSAMPLE], s_p[q * OVERSAMPLE])) lo = q;
    }
    bkt[r] = lo;
    rank[r] = le < tile_n ? atomicAdd(&s_cnt[lo], 1u) : 0u;
  }
  __syncthreads();
  // Exclusive scan of the tile's bucket counts (the first B threads).
  uint32_t c = tid < (uint32_t)B ? s_cnt[tid] : 0u;
  uint32_t x = c;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, WAVE);
    if (lane_id() >= off) x += y;
  }
  if (lane_id() == WAVE - 1) s_w[tid / WAVE] = x;
  __syncthreads();
  uint32_t* row = fa.words + FRONT_OFFS + blockIdx.x * (uint32_t)(B + 1);
  if (tid < (uint32_t)B) {
    uint32_t before = 0;
    for (uint32_t w = 0; w < tid / WAVE; ++w) before += s_w[w];
    s_off[tid] = before + x - c;
    row[tid] = before + x - c;
    if (tid == 0) row[B] = tile_n;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t le = (uint32_t)r * FT + tid;
    if (le < tile_n) {
      const uint32_t dst = tile0 + s_off[bkt[r]] + rank[r];
      fa.tmp_keys[dst] = ek[r];
      fa.tmp_ties[dst] = ep[r];
      if constexpr (BATCH) found[tile0 + le] = 1;  // the answers' default
    }
  }
}

// ------------------------------------------------------------------ bucket sort
// The bucket's m elements (in s_k, s_p) into sorted order, written to the batch's sorted arrays
// from position start, and back to s_k for the summary.
template <int E>
STM_DEV void sort_bucket(const FrontArgs& fa, uint32_t m, uint32_t start, uint64_t* s_k, uint32_t* s_p,
                         BinShared& s_bin, BucketSum& sum, Acc* s_acc) {
  const uint32_t tid = threadIdx.x;
  uint64_t k[E];
  uint32_t p[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    k[r] = i < m ? s_k[i] : KEY_EMPTY;
    p[r] = i < m ? s_p[i] : ~0u;
  }
  bin_sort<FT, E>(m, k, p, s_k, s_p, s_bin);
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    const bool v = i < m;
    const uint64_t key = s_k[i];
    const uint32_t tie = s_p[i];
    if (v) {
      const_cast<uint64_t*>(fa.fold.skeys)[start + i] = key;
      const_cast<uint32_t*>(fa.fold.sidx)[start + i] = payload_of(tie);
    }
    const uint64_t hm = ballot(v && i > 0 && s_k[i > 0 ? i - 1 : 0] != key);
    const uint64_t im = ballot(v && (tie & 3u) == OP_INSERT && key != KEY_EMPTY);
    const uint32_t c = (uint32_t)r * FW + tid / WAVE;
    if (lane_id() == 0) s_acc[c] = acc_round(acc_identity(), hm, im, start + c * WAVE);
  }
  __syncthreads();
  if (tid < (uint32_t)WAVE)
    sum.acc = wave_combine(tid < (uint32_t)(FW * E) ? s_acc[tid] : acc_identity());
}

// Bucket blockIdx.x of B: its pieces, one per tile of tile_ops elements, into LDS, sorted there.
__global__ __launch_bounds__(FT) void k_front_bucket(FrontArgs fa, uint32_t tile_ops, uint32_t B) {
  __shared__ uint64_t s_k[BUCKET_CAP];
  __shared__ uint32_t s_p[BUCKET_CAP];
  __shared__ uint32_t s_src[TILES_MAX], s_dst[TILES_MAX], s_len[TILES_MAX];
  __shared__ uint32_t s_w[2][2];
  __shared__ Acc s_acc[BUCKET_CAP / WAVE];
  __shared__ BinShared s_bin;
  static_assert(BUCKET_CAP / WAVE <= WAVE, "one wavefront combines a bucket's states");
  static_assert(TILES_MAX <= 2 * WAVE, "the tiles fit two wavefronts");
  const uint32_t n = front_in(fa).n;
  const uint32_t b = blockIdx.x;
  const uint32_t tid = threadIdx.x;
  const uint32_t tiles = (n + tile_ops - 1) / tile_ops;
  BucketSum* sums = reinterpret_cast<BucketSum*>(fa.words + FRONT_SUMS);
  uint32_t o0 = 0, len = 0, x = 0, y = 0;
  if (tid < 2 * WAVE) {
    if (tid < tiles) {
      const uint32_t* row = fa.words + FRONT_OFFS + tid * (B + 1) + b;
      o0 = row[0];
      len = row[1] - o0;
    }
    x = len;
    y = o0;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const uint32_t xs = __shfl_up(x, off, WAVE), ys = __shfl_up(y, off, WAVE);
      if (lane_id() >= off) {
        x += xs;
        y += ys;
      }
    }
    if (lane_id() == WAVE - 1) {
      s_w[tid / WAVE][0] = x;
      s_w[tid / WAVE][1] = y;
    }
  }
  __syncthreads();
  const uint32_t m = s_w[0][0] + s_w[1][0];
  const uint32_t start = s_w[0][1] + s_w[1][1];  // elements of the buckets before this one
  if (tid < tiles) {
    s_src[tid] = tid * tile_ops + o0;
    s_dst[tid] = x - len + (tid >= WAVE ? s_w[0][0] : 0u);
    s_len[tid] = len;
  }
  __syncthreads();
  BucketSum sum{start, acc_identity()};
  if (m > BUCKET_CAP) {
    if (tid == 0) *fa.retry = 1;
  } else if (m > 0) {
    bin_sort_open<FT>(s_bin);
    // Eight lanes per piece: the mean piece is a few elements.
    for (uint32_t t = tid / 8; t < tiles; t += FT / 8) {
      const uint32_t src = s_src[t], dst = s_dst[t], l = s_len[t];
      for (uint32_t q = tid & 7u; q < l; q += 8) {
        s_k[dst + q] = fa.tmp_keys[src + q];
        s_p[dst + q] = fa.tmp_ties[src + q];
      }
    }
    __syncthreads();
    if (m <= FT) sort_bucket<1>(fa, m, start, s_k, s_p, s_bin, sum, s_acc);
    else if (m <= 2 * FT) sort_bucket<2>(fa, m, start, s_k, s_p, s_bin, sum, s_acc);
    else sort_bucket<4>(fa, m, start, s_k, s_p, s_bin, sum, s_acc);
  }
  if (tid == 0) sums[b] = sum;
}

// ------------------------------------------------------------------ fold of a bucket
__global__ __launch_bounds__(FT) void k_front_fold(FrontArgs fa, uint32_t B) {
  __shared__ Acc s_acc[FW];
  FoldArgs a = fa.fold;
  fold_resolve(a);
  const uint32_t n = a.n;
  if (n == 0) return;  // k_front_split left empty counters
  const uint32_t b = blockIdx.x;
  const uint32_t tid = threadIdx.x;
  const uint32_t wave = tid / WAVE;
  if (*fa.retry) {
    if (b == 0 && tid == 0) a.counters->sort_retry = 1;  // no groups: the batch runs empty
    return;
  }
  const BucketSum* sums = reinterpret_cast<const BucketSum*>(fa.words + FRONT_SUMS);
  // State before the bucket: the other buckets' summaries, each completed by whether its first
  // element starts a group.  The first bucket sums all of them for the number of groups instead.
  Acc v = acc_identity();
  const uint32_t start = sums[b].start;
  const uint32_t end = b + 1 < B ? sums[b + 1].start : n;
  if (tid < B && (tid < b || b == 0)) {
    const BucketSum q = sums[tid];
    const uint32_t qe = tid + 1 < B ? sums[tid + 1].start : n;
    if (qe > q.start) {
      v = q.acc;
      if (q.start == 0 || a.skeys[q.start > 0 ? q.start - 1 : 0] != a.skeys[q.start]) {
        v.c += 1;
        v.head = v.head >= 0 ? v.head : (int32_t)q.start;
        v.m &= ~ACC_LEAD;
      }
    }
  }
  v = wave_combine(v);
  if (lane_id() == 0) s_acc[wave] = v;
  __syncthreads();
  Acc carry = acc_identity();
#pragma unroll
  for (int w = 0; w < (int)(BUCKETS_MAX / WAVE); ++w) carry = acc_combine(carry, s_acc[w]);
  if (b == 0) {
    if (tid == 0) {
      a.counters->n_unique = carry.c;
      a.counters->n_upserts = carry.m & ~ACC_LEAD;
    }
    carry = acc_identity();
  }
  __syncthreads();
  for (uint32_t r0 = start; r0 < end; r0 += FT) {
    const uint32_t i = r0 + tid;
    FoldElem x;
    x.valid = i < end;
    x.i = (int32_t)i;
    const uint32_t ic = min(i, end - 1);  // unconditional loads from a clamped index
    const uint64_t prev = a.skeys[ic > 0 ? ic - 1 : 0];
    const uint64_t next = a.skeys[min(ic + 1, n - 1)];
    x.key = a.skeys[ic];
    const uint32_t pl = a.sidx[ic];
    x.pos = pos_of(pl);
    x.ins = x.valid && op_of(pl) == OP_INSERT && x.key != KEY_EMPTY;
    x.end = x.valid && (i + 1 == n || next != x.key);
    const uint64_t hm = ballot(x.valid && (i == 0 || prev != x.key)), im = ballot(x.ins);
    const uint32_t rb = r0 + wave * WAVE;
    if (lane_id() == 0) s_acc[wave] = acc_round(acc_identity(), hm, im, rb);
    __syncthreads();
    Acc before = carry;
#pragma unroll
    for (int w = 0; w < FW; ++w) {
      const Acc t = s_acc[w];
      if ((uint32_t)w < wave) before = acc_combine(before, t);
      carry = acc_combine(carry, t);
    }
    fold_place(x, hm, im, rb, before);
    x.lb_pos = x.valid && x.lb >= 0 ? pos_of(a.sidx[x.lb]) : 0u;
    fold_gather(a, x);
    fold_store(a, x, &a.counters->n_bad);
    __syncthreads();
  }
}

// ------------------------------------------------------------------ launcher
template <int E, int S, bool BATCH>
static hipError_t launch_shape(const FrontArgs& a, uint32_t n_max, hipStream_t s) {
  constexpr uint32_t B = S / OVERSAMPLE;
  const uint32_t tile = FT * E;
  k_front_split<E, S, BATCH><<<(n_max + tile - 1) / tile, FT, 0, s>>>(a);
  k_front_bucket<<<B, FT, 0, s>>>(a, tile, B);
  if constexpr (BATCH) k_front_fold<<<B, FT, 0, s>>>(a, B);
  return hipGetLastError();
}

// About 512 ops per bucket: a bucket then mostly sorts in one element per thread.
template <bool BATCH>
static hipError_t launch_split(const FrontArgs& a, uint32_t n, hipStream_t s) {
  if (n <= (1u << 14)) return launch_shape<1, 256, BATCH>(a, n, s);
  if (n <= (1u << 15)) return launch_shape<1, 512, BATCH>(a, n, s);
  if (n <= (1u << 16)) return launch_shape<1, 1024, BATCH>(a, n, s);
  return launch_shape<2, 2048, BATCH>(a, n, s);
}

// a.fold.n is the op count, or with a.fold.desc the largest count (at most FRONT_MAX_OPS).
hipError_t front_batch(FrontArgs a, hipStream_t s) {
  const uint32_t n = a.fold.n;
  if (n == 0) return hipSuccess;
  if (n > FRONT_MAX_OPS) return hipErrorInvalidValue;
  a.retry = a.words + FRONT_RETRY;
  if (n <= FT) {
    k_front_small<1><<<1, FT, 0, s>>>(a);
    return hipGetLastError();
  }
  if (n <= FRONT_SMALL) {
    k_front_small<2><<<1, FT, 0, s>>>(a);
    return hipGetLastError();
  }
  return launch_split<true>(a, n, s);
}

size_t front_sort_words(uint32_t n) {
  if (n <= FRONT_SMALL) return 0;
  const uint32_t tiles = n <= (1u << 16) ? (n + FT - 1) / FT : (n + 2 * FT - 1) / (2 * FT);
  const uint32_t B = n <= (1u << 14) ? 32u : n <= (1u << 15) ? 64u : n <= (1u << 16) ? 128u : 256u;
  return FRONT_OFFS + (size_t)tiles * (B + 1);
}

// Stable sort of fs.n keys.  *fs.need is 1 afterwards where a bucket overflowed, and the output then
// incomplete.  stm_sort_pairs_device with the normalized radix passes and their dozen launches, before
// its allocations became one, and now: 1000 keys 95 / 36 µs, 16384 keys 103 / 48, 2^18 keys 145 / 95.
hipError_t front_sort(const FrontSort& fs, hipStream_t s) {
  if (fs.n == 0) return hipSuccess;
  if (fs.n > FRONT_MAX_OPS) return hipErrorInvalidValue;
  if (fs.n <= FT) {
    k_front_keys<1><<<1, FT, 0, s>>>(fs);
    return hipGetLastError();
  }
  if (fs.n <= FRONT_SMALL) {
    k_front_keys<2><<<1, FT, 0, s>>>(fs);
    return hipGetLastError();
  }
  FrontArgs a{};
  a.keys = fs.keys;
  a.fold.n = fs.n;
  a.fold.skeys = fs.keys_out;
  a.fold.sidx = fs.idx_out;
  a.tmp_keys = fs.tmp_keys;
  a.tmp_ties = fs.tmp_ties;
  a.words = fs.words;
  a.retry = fs.need;
  a.stall = fs.stall;
  a.barrier = fs.barrier;
  return launch_split<false>(a, fs.n, s);
}

}  // namespace stm
