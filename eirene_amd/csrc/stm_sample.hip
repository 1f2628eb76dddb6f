// stm_sample.hip — stable sort of SAMPLE_SORT_MIN .. SAMPLE_SORT_MAX (key, position) pairs by
// sampled buckets: the batch is read twice and written twice, where the normalized radix form of
// stm_sort.hip takes a range pass, three digit passes of two reads each and a fix-up pass.
//
//   k_sample_fetch   (above 4096 samples) gathers the samples' keys
//   k_sample_pick    sorts S = 8 B samples of the batch (one per equal stretch of the input, at a
//                    hashed place); every 8th is a splitter
//   k_sample_split   one workgroup per tile orders the tile by bucket (binary search of the B
//                    splitters in LDS), and notes where each bucket begins in it
//   k_sample_bucket  one workgroup per bucket collects its pieces from the tiles, sorts them in LDS
//                    by exact (key, position) and writes them to their final place
//
// Buckets are cut between samples of (key, position), so the ops of a hot key are shared by as many
// buckets as they fill and no normalization is needed.  A bucket holds 1024 elements in the mean
// (2048 above 2^21); one with more than BUCKET_CAP is taken in groups of the eight intervals between
// its own samples, and an interval (an eighth of a bucket in the mean) that holds more, as happens
// about once in 500 batches of the largest size, in halves of its key range.  Only a half that
// is still too large, which takes keys built to mislead the sample, asks for the exact sort.
//
// Bound by the round trips of a workgroup (k_sample_pick: 4 to 16 workgroups on the chip;
// k_sample_bucket: about 13 µs of row words, elements and barriers per bucket, two buckets on a CU) and,
// in k_sample_split, by one tile per CU at a time.  Sort kernels, normalized radix / this: 2^20 keys
// 91 / 55 µs, 2^22 keys 168 / 134 (fetch 3, pick 17, split 45, bucket 64, exact-sort check 5).  Whole
// calls on 2^20 uniform keys with 5 % inserts: 2^19 ops 152 / 114 µs, 2^20 182 / 148, 2^21 238 / 213, 2^22
// 405 / 376; lookups of Zipf keys on 2^22 keys: 2^19 ops 226 / 127, 2^20 256 / 162, 2^22 547 / 376.
#include <algorithm>

#include "stm_binsort.hpp"
#include "stm_common.hpp"
#include "stm_internal.hpp"

namespace stm {

constexpr uint32_t PER_BUCKET = 8;         // samples per bucket
constexpr uint32_t PART_CAP = 2 * FT;      // samples one workgroup of k_sample_pick sorts (FT in the mean)
constexpr uint32_t BUCKET_CAP = 4 * FT;    // elements of a bucket sorted at once
constexpr uint32_t TILES_MAX = 256;
constexpr uint32_t BUCKETS_MAX = 2048;

// Scratch (u32 words from the given base, 8-byte aligned): the samples' keys and ties in order,
// the splitters' keys and ties, a word per workgroup of k_sample_pick (1: too many samples met in
// it), then the tiles' bucket bounds (u16).
struct SampleScratch {
  uint64_t* skey;
  uint64_t* bkey;
  uint32_t* stie;
  uint32_t* btie;
  uint32_t* over;
  uint16_t* rows;
};
static size_t sample_words_of(uint32_t B) {
  return 3 * (size_t)(PER_BUCKET + 1) * B + 64 + ((size_t)TILES_MAX * (B + 1) + 1) / 2;
}
static SampleScratch sample_scratch(uint32_t* words, uint32_t B) {
  SampleScratch s;
  s.skey = reinterpret_cast<uint64_t*>(words);
  s.bkey = s.skey + PER_BUCKET * B;
  s.stie = reinterpret_cast<uint32_t*>(s.bkey + B);
  s.btie = s.stie + PER_BUCKET * B;
  s.over = s.btie + B;
  s.rows = reinterpret_cast<uint16_t*>(s.over + 64);
  return s;
}

// ------------------------------------------------------------------ samples
// Input position of sample j of S.
template <int S>
STM_DEV uint32_t sample_place(uint32_t j, uint32_t n) {
  const uint32_t lo = (uint32_t)((uint64_t)j * n / S);
  const uint32_t hi = (uint32_t)((uint64_t)(j + 1) * n / S);
  return min(lo + (uint32_t)(((uint64_t)hash32(j) * (hi - lo)) >> 32), n - 1);
}

// Sample j's key to raw[j % G * FT + j / G] (G = S / FT), where k_sample_pick reads it in order.  A
// launch of its own above 4096 samples: one CU fetches scattered lines at 2.6 clocks each, so that
// k_sample_pick took 30 µs with 16384 samples fetched by itself (each of its workgroups reads all).
template <int S>
__global__ __launch_bounds__(256) void k_sample_fetch(const uint64_t* __restrict__ keys, uint32_t n,
                                                      uint64_t* __restrict__ raw) {
  constexpr uint32_t G = S / FT;
  const uint32_t j = blockIdx.x * 256 + threadIdx.x;
  if (j < (uint32_t)S) raw[j % G * FT + j / G] = gload(keys + sample_place<S>(j, n));
}

// Workgroup g of S / FT sorts the samples of its part of the key range: it reads all S (in one round
// trip; from raw, or from the batch where raw is null), cuts the range at every (S / FT)-th of FT of
// them, which it sorts first, and keeps those of its own part, FT in the mean.  Its first sample's
// rank is the number of samples below.  One launch, where a sort of S elements by one workgroup does
// not fit the LDS.  Workgroup 0 clears the control words.
template <int S>
__global__ __launch_bounds__(FT) void k_sample_pick(const uint64_t* __restrict__ keys,
                                                    const uint64_t* __restrict__ raw, uint32_t n,
                                                    SampleScratch sc, uint32_t* __restrict__ stall,
                                                    uint32_t* __restrict__ barrier) {
  constexpr int G = S / FT;
  static_assert(G >= 1 && G <= 64, "one word of `over` per workgroup");
  __shared__ uint64_t s_k[PART_CAP];
  __shared__ uint32_t s_p[PART_CAP];
  __shared__ BinShared s_bin;
  __shared__ uint32_t s_n, s_below;
  const uint32_t tid = threadIdx.x, g = blockIdx.x;
  if (g == 0 && tid == 0) {
    *stall = 0;
    *barrier = 0;
  }
  auto place = [&](uint32_t j) { return sample_place<S>(j, n); };
  uint64_t k[G];
#pragma unroll
  for (int r = 0; r < G; ++r)
    k[r] = raw ? gload(raw + r * FT + tid) : gload(keys + place(tid * (uint32_t)G + (uint32_t)r));
  uint64_t k1[1];
  uint32_t p1[1];
  k1[0] = k[0];
  p1[0] = place(tid * (uint32_t)G) << 2;
  bin_sort_open<FT>(s_bin);
  if (tid == 0) {
    s_n = 0;
    s_below = 0;
  }
  __syncthreads();
  bin_sort<FT, 1>(FT, k1, p1, s_k, s_p, s_bin);
  const uint32_t cl = g * (FT / G), ch = min((g + 1) * (FT / G), (uint32_t)FT - 1);
  const uint64_t lk = s_k[cl], hk = s_k[ch];
  const uint32_t lp = s_p[cl], hp = s_p[ch];
  __syncthreads();
  bin_sort_open<FT>(s_bin);
  uint32_t n_below = 0;
#pragma unroll
  for (int r = 0; r < G; ++r) {
    const uint32_t p = place(tid * (uint32_t)G + (uint32_t)r) << 2;
    const bool below = g > 0 && elem_less(k[r], p, lk, lp);
    const bool keep = !below && (g + 1 == (uint32_t)G || elem_less(k[r], p, hk, hp));
    n_below += (uint32_t)__popcll(ballot(below));
    if (keep) {
      const uint32_t at = atomicAdd(&s_n, 1u);
      if (at < PART_CAP) {
        s_k[at] = k[r];
        s_p[at] = p;
      }
    }
  }
  if (lane_id() == 0 && n_below) atomicAdd(&s_below, n_below);
  __syncthreads();
  const uint32_t m = s_n, first = s_below;
  if (tid == 0) sc.over[g] = m > PART_CAP ? 1u : 0u;
  if (m > PART_CAP) return;
  uint64_t k2[2];
  uint32_t p2[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    k2[r] = i < m ? s_k[i] : KEY_EMPTY;
    p2[r] = i < m ? s_p[i] : ~0u;
  }
  bin_sort<FT, 2>(m, k2, p2, s_k, s_p, s_bin);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    if (i < m) {
      const uint32_t q = first + i;
      sc.skey[q] = s_k[i];
      sc.stie[q] = s_p[i];
      if (q % PER_BUCKET == 0) {
        sc.bkey[q / PER_BUCKET] = s_k[i];
        sc.btie[q / PER_BUCKET] = s_p[i];
      }
    }
  }
}

// ------------------------------------------------------------------ split
// Tile blockIdx.x of FT * E elements, ordered by bucket (in any order within one) through LDS so
// that the stores are coalesced.  The splitters' ties are read only for keys equal to a splitter's.
template <int E, int B>
__global__ __launch_bounds__(FT) void k_sample_split(const uint64_t* __restrict__ keys,
                                                     const uint8_t* __restrict__ ops, uint32_t n,
                                                     SampleScratch sc, uint32_t* __restrict__ need,
                                                     uint64_t* __restrict__ tmp_keys,
                                                     uint32_t* __restrict__ tmp_ties,
                                                     uint8_t* __restrict__ found) {
  constexpr uint32_t TILE = FT * E;
  constexpr int PER = B > FT ? B / FT : 1;  // buckets per thread of the scan
  __shared__ uint64_t s_stage[TILE];
  __shared__ uint64_t s_spl[B];
  __shared__ uint32_t s_cnt[B];  // counts, then first places within the tile
  __shared__ uint32_t s_w[FW];
  const uint32_t tid = threadIdx.x;
  const uint32_t tile0 = blockIdx.x * TILE;
  const uint32_t tile_n = min(TILE, n - tile0);
  uint64_t k[E];
  uint32_t op[(E + 15) / 16];
#pragma unroll
  for (int q = 0; q < (E + 15) / 16; ++q) op[q] = 0;
#pragma unroll
  for (int r = 0; r < E; ++r) k[r] = gload(keys + tile0 + min((uint32_t)r * FT + tid, tile_n - 1));
  if (ops) {
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const uint32_t o = gload(ops + tile0 + min((uint32_t)r * FT + tid, tile_n - 1));
      op[r / 16] |= (o > 3u ? 1u : o) << (2 * (r % 16));
    }
  }
  for (uint32_t q = tid; q < (uint32_t)B; q += FT) {
    s_spl[q] = sc.bkey[q];
    s_cnt[q] = 0;
  }
  if (blockIdx.x == 0 && tid < (uint32_t)WAVE) {  // the sort's request for the exact passes
    const bool over = tid < PER_BUCKET * B / FT && sc.over[tid] != 0;
    const uint64_t any = ballot(over);
    if (tid == 0) *need = any ? 1u : 0u;
  }
  __syncthreads();
  auto tie = [&](int r) {
    return ((tile0 + (uint32_t)r * FT + tid) << 2) | ((op[r / 16] >> (2 * (r % 16))) & 3u);
  };
  uint32_t at[E];  // bucket in the upper half, place within the tile's part of it in the lower
#pragma unroll
  for (int r = 0; r < E; ++r) {
    uint32_t lo = 0;
#pragma unroll
    for (int step = B / 2; step > 0; step >>= 1) {
      const uint32_t q = lo + (uint32_t)step;
      const uint64_t sk = s_spl[q];
      bool right = sk < k[r];
      if (sk == k[r]) right = sc.btie[q] <= tie(r);
      lo = right ? q : lo;
    }
    const bool v = (uint32_t)r * FT + tid < tile_n;
    at[r] = (lo << 16) | (v ? atomicAdd(&s_cnt[lo], 1u) : 0u);
  }
  __syncthreads();
  // Exclusive scan of the counts.
  uint32_t c[PER], sum = 0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    c[q] = tid * PER + q < (uint32_t)B ? s_cnt[tid * PER + q] : 0u;
    sum += c[q];
  }
  uint32_t x = sum;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, WAVE);
    if (lane_id() >= off) x += y;
  }
  if (lane_id() == WAVE - 1) s_w[tid / WAVE] = x;
  __syncthreads();
  uint32_t run = x - sum;
#pragma unroll
  for (uint32_t w = 0; w < (uint32_t)FW; ++w) run += w < tid / WAVE ? s_w[w] : 0u;
  uint16_t* row = sc.rows + (size_t)blockIdx.x * (B + 1);
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    if (tid * PER + q < (uint32_t)B) {
      s_cnt[tid * PER + q] = run;
      row[tid * PER + q] = (uint16_t)run;
    }
    run += c[q];
  }
  if (tid == 0) row[B] = (uint16_t)tile_n;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    at[r] = s_cnt[at[r] >> 16] + (at[r] & 0xffffu);
    if ((uint32_t)r * FT + tid < tile_n) s_stage[at[r]] = k[r];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    if (i < tile_n) tmp_keys[tile0 + i] = s_stage[i];
  }
  __syncthreads();
  uint32_t* s_tie = reinterpret_cast<uint32_t*>(s_stage);
#pragma unroll
  for (int r = 0; r < E; ++r)
    if ((uint32_t)r * FT + tid < tile_n) s_tie[at[r]] = tie(r);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const uint32_t i = (uint32_t)r * FT + tid;
    if (i < tile_n) {
      tmp_ties[tile0 + i] = s_tie[i];
      if (found) found[tile0 + i] = 1;  // the answers' default
    }
  }
}

// ------------------------------------------------------------------ buckets
// One bucket of B.  Consecutive buckets share the lines of their pieces, so they go to the same
// XCD (workgroups are dealt to the eight XCDs in turn).
// The elements go from memory into registers (thread i takes element i of the pieces laid end to
// end, which it finds by binary search: balanced also where the input is sorted and a bucket is one
// long piece), are counted into bins by the leading bits of their distance from the bucket's
// splitter, written to LDS bin by bin, and ranked within their bin as they leave it: one trip
// through the LDS, and the stores to the output are within a bin's length of coalesced.  Bins hold
// an element or two; keys that crowd one (medium-hot keys) cost a comparison per pair, which beats
// a comparison sort of the bucket up to some thousand equal keys.
// A bucket of more than BUCKET_CAP elements is taken in groups of consecutive intervals between its
// own samples, each group collected in LDS first.
__global__ __launch_bounds__(FT, 8) void k_sample_bucket(uint32_t n, uint32_t tile_ops, uint32_t B,
                                                                 SampleScratch sc,
                                                                 const uint64_t* __restrict__ tmp_keys,
                                                                 const uint32_t* __restrict__ tmp_ties,
                                                                 uint64_t* __restrict__ keys_out,
                                                                 uint32_t* __restrict__ idx_out,
                                                                 uint32_t* __restrict__ need) {
  constexpr int E = BUCKET_CAP / FT;
  constexpr int WORDS = E / 2;  // of s_place, per thread
  constexpr uint32_t PER = BINS / FT;
  constexpr uint32_t NW = FW;
  __shared__ uint64_t s_k[BUCKET_CAP];
  __shared__ uint32_t s_p[BUCKET_CAP];
  __shared__ uint32_t s_src[TILES_MAX], s_dst[TILES_MAX];  // s_src: less s_dst
  __shared__ uint32_t s_w[TILES_MAX / WAVE][2];
  __shared__ uint32_t s_sub[PER_BUCKET], s_fill;
  __shared__ BinShared s_bin;
  // For crowded bins: elements below (low half) and above (high half) the middle key, by bin;
  // counts, then prefixes, of the places, two to a word; the range of ties.
  __shared__ uint32_t s_side[BINS], s_place[BUCKET_CAP / 2], s_tmin, s_tmax;
  const uint32_t tid = threadIdx.x, wave = tid / WAVE;
  const uint32_t b = (blockIdx.x & 7u) * (B / 8) + blockIdx.x / 8;
  const uint32_t tiles = (n + tile_ops - 1) / tile_ops;
  uint32_t o0 = 0, len = 0, x = 0, y = 0;
  if (tid < TILES_MAX) {
    if (tid < tiles) {
      const uint16_t* row = sc.rows + (size_t)tid * (B + 1) + b;
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
      s_w[wave][0] = x;
      s_w[wave][1] = y;
    }
  }
  if (tid < PER_BUCKET) s_sub[tid] = 0;
  const uint64_t* bk = sc.skey + PER_BUCKET * b;  // the bucket's samples
  const uint32_t* bt = sc.stie + PER_BUCKET * b;
  // Its bounds travel with the row's words (the last bucket has no upper one).
  const uint32_t past = b + 1 == B ? PER_BUCKET - 1 : PER_BUCKET;
  const uint64_t blo = uniform64(bk[0]), bhi = uniform64(bk[past]);
  const uint32_t btlo = uniform32(bt[0]), bthi = uniform32(bt[past]);
  __syncthreads();
  uint32_t m = 0, start = 0, before = 0;  // start: elements of the buckets below
#pragma unroll
  for (uint32_t w = 0; w < TILES_MAX / WAVE; ++w) {
    before += w < wave ? s_w[w][0] : 0u;
    m += s_w[w][0];
    start += s_w[w][1];
  }
  m = uniform32(m);
  start = uniform32(start);
  if (tid < TILES_MAX) {
    s_dst[tid] = before + x - len;
    s_src[tid] = tid * tile_ops + o0 - (before + x - len);
  }
  __syncthreads();
  if (m == 0) return;
  // Where element i of the bucket lies: in the last piece that begins at or before it.
  auto source = [&](uint32_t i) {
    uint32_t t = 0;
#pragma unroll
    for (uint32_t step = TILES_MAX / 2; step > 0; step >>= 1) t = s_dst[t + step] <= i ? t + step : t;
    return s_src[t] + i;
  };
  auto interval = [&](uint64_t k, uint32_t p) {
    uint32_t i = 0;
    for (uint32_t q = 1; q < PER_BUCKET; ++q) i += elem_less(k, p, bk[q], bt[q]) ? 0u : 1u;
    return i;
  };
  const bool one = m <= BUCKET_CAP;
  if (!one) {
    for (uint32_t i = tid; i < m; i += FT) {
      const uint32_t src = source(i);
      atomicAdd(&s_sub[interval(tmp_keys[src], tmp_ties[src])], 1u);
    }
    __syncthreads();
  }
  // An interval of its own that is too large is cut once more, between its bounds.
  uint32_t half = 0, upper = 0;  // half 1, 2: the pass takes the elements below (mk, mt), the others
  uint64_t mk = 0;
  uint32_t mt = 0;
#pragma unroll 1
  for (uint32_t i0 = 0, i1; i0 < PER_BUCKET; i0 = half == 1 ? i0 : i1) {
    uint32_t gm = one ? m : uniform32(s_sub[i0]);
    i1 = one ? PER_BUCKET : i0 + 1;
    if (half == 1) {
      half = 2;
      gm = upper;
    } else {
      half = 0;
      while (i1 < PER_BUCKET && gm + uniform32(s_sub[i1]) <= BUCKET_CAP) gm += uniform32(s_sub[i1++]);
      if (gm > BUCKET_CAP && !(b == 0 && i0 == 0) && !(b + 1 == B && i1 == PER_BUCKET)) {
        const uint64_t k0 = uniform64(bk[i0]), k1 = uniform64(bk[i1]);
        const uint32_t t0 = uniform32(bt[i0]), t1 = uniform32(bt[i1]);
        mk = k0 + (k1 - k0) / 2;
        mt = k0 == k1 ? t0 + (t1 - t0) / 2 : 0u;
        __syncthreads();
        if (tid == 0) s_fill = 0;
        __syncthreads();
        for (uint32_t i = tid; i < m; i += FT) {
          const uint32_t src = source(i);
          const uint64_t key = tmp_keys[src];
          const uint32_t t = tmp_ties[src];
          if (interval(key, t) == i0 && elem_less(key, t, mk, mt)) atomicAdd(&s_fill, 1u);
        }
        __syncthreads();
        half = 1;
        upper = gm - uniform32(s_fill);
        gm -= upper;
      }
    }
    const uint32_t out = start;
    start += gm;
    if (gm == 0) continue;
    if (gm > BUCKET_CAP) {
      if (tid == 0) *need = 1;
      continue;
    }
    __syncthreads();  // the group before has left the LDS
    for (uint32_t q = tid; q < BINS; q += FT) s_bin.bin[q] = 0;
    if (tid == 0) {
      s_fill = 0;
      s_bin.mn = KEY_EMPTY;
      s_bin.mx = 0;
      s_bin.heavy = 0;
    }
    __syncthreads();
    uint64_t k[E];
    uint32_t p[E], at[E];
    if (one) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        const uint32_t i = (uint32_t)r * FT + tid;
        k[r] = KEY_EMPTY;
        p[r] = ~0u;
        if (i < gm) {
          const uint32_t src = source(i);
          k[r] = gload(tmp_keys + src);
          p[r] = gload(tmp_ties + src);
        }
      }
    } else {
      for (uint32_t i = tid; i < m; i += FT) {
        const uint32_t src = source(i);
        const uint64_t key = tmp_keys[src];
        const uint32_t t = tmp_ties[src];
        const uint32_t v = interval(key, t);
        if (v >= i0 && v < i1 && (half == 0 || elem_less(key, t, mk, mt) == (half == 1))) {
          const uint32_t to = atomicAdd(&s_fill, 1u);
          s_k[to] = key;
          s_p[to] = t;
        }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < E; ++r) {
        const uint32_t i = (uint32_t)r * FT + tid;
        k[r] = i < gm ? s_k[i] : KEY_EMPTY;
        p[r] = i < gm ? s_p[i] : ~0u;
      }
    }
    // The group's bounds: its samples', or the elements' own where it is open at one end.
    const bool last = i1 == PER_BUCKET && b + 1 == B;
    uint64_t klo = blo, khi = bhi;
    uint32_t tlo = btlo, thi = bthi;
    if (!one) {
      const uint32_t end = last ? past : i1;
      klo = uniform64(bk[i0]);
      khi = uniform64(bk[end]);
      tlo = uniform32(bt[i0]);
      thi = uniform32(bt[end]);
      if (half) {
        if (klo == khi) (half == 1 ? thi : tlo) = mt;
        else (half == 1 ? khi : klo) = mk;
      }
    }
    if (last || (b == 0 && i0 == 0)) {
      uint64_t mn = KEY_EMPTY, mx = 0;
#pragma unroll
      for (int r = 0; r < E; ++r) {
        if ((uint32_t)r * FT + tid < gm) {
          mn = k[r] < mn ? k[r] : mn;
          mx = k[r] > mx ? k[r] : mx;
        }
      }
#pragma unroll
      for (int off = 1; off < WAVE; off <<= 1) {
        const uint64_t u = shfl64(mn, lane_id() ^ off), v = shfl64(mx, lane_id() ^ off);
        mn = u < mn ? u : mn;
        mx = v > mx ? v : mx;
      }
      if (lane_id() == 0) {
        atomicMin((unsigned long long*)&s_bin.mn, (unsigned long long)mn);
        atomicMax((unsigned long long*)&s_bin.mx, (unsigned long long)mx);
      }
      __syncthreads();
      klo = uniform64(s_bin.mn);
      khi = uniform64(s_bin.mx);
      tlo = 0;
      thi = ~0u;
    }
    // Bin: leading bits of the distance from the lower bound, of the tie where all keys are equal.
    const bool same = klo == khi;
    const uint64_t base = same ? (uint64_t)tlo : klo;
    const uint64_t range = same ? (uint64_t)(thi - tlo) : khi - klo;
    const uint32_t bits = range ? 64u - (uint32_t)__clzll((long long)range) : 0u;
    const uint32_t shift = bits > BIN_BITS ? bits - BIN_BITS : 0u;
    auto bin_of = [&](uint64_t key, uint32_t t) {
      const uint64_t d = ((same ? (uint64_t)t : key) - base) >> shift;
      return (uint32_t)min<uint64_t>(d, BINS - 1);
    };
#pragma unroll
    for (int r = 0; r < E; ++r) {
      at[r] = 0;
      if ((uint32_t)r * FT + tid < gm) {
        at[r] = atomicAdd(&s_bin.bin[bin_of(k[r], p[r])], 1u);
        if (at[r] >= BIN_MAX) s_bin.heavy = 1;
      }
    }
    __syncthreads();
    const bool heavy = uniform32(s_bin.heavy) != 0;
    // Exclusive scan of the bins, PER per thread.
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      c[q] = s_bin.bin[tid * PER + q];
      sum += c[q];
    }
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const uint32_t z = __shfl_up(incl, off, WAVE);
      if (lane_id() >= off) incl += z;
    }
    if (lane_id() == WAVE - 1) s_bin.w[wave] = incl;
    __syncthreads();
    uint32_t run = incl - sum;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) run += w < wave ? s_bin.w[w] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      s_bin.bin[tid * PER + q] = run;
      run += c[q];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) {
      if ((uint32_t)r * FT + tid < gm) {
        at[r] += s_bin.bin[bin_of(k[r], p[r])];
        s_k[at[r]] = k[r];
        s_p[at[r]] = p[r];
      }
    }
    if (heavy) {
      for (uint32_t q = tid; q < BINS; q += FT) s_side[q] = 0;
      for (uint32_t q = tid; q < BUCKET_CAP / 2; q += FT) s_place[q] = 0;
      if (tid == 0) {
        s_tmin = ~0u;
        s_tmax = 0;
      }
    }
    __syncthreads();
    auto bin_end = [&](uint32_t bin) { return bin + 1 < BINS ? s_bin.bin[bin + 1] : gm; };
    auto rank_in = [&](uint32_t lo, uint32_t hi, uint64_t key, uint32_t t) {
      uint32_t to = lo;
      if (hi - lo > 1)
        for (uint32_t j = lo; j < hi; ++j) to += elem_less(s_k[j], s_p[j], key, t) ? 1u : 0u;
      return to;
    };
    if (!heavy) {
#pragma unroll
      for (int r = 0; r < E; ++r) {
        const uint32_t i = (uint32_t)r * FT + tid;
        if (i < gm) {
          const uint64_t key = s_k[i];
          const uint32_t t = s_p[i];
          const uint32_t bin = bin_of(key, t);
          const uint32_t to = rank_in(s_bin.bin[bin], bin_end(bin), key, t);
          keys_out[out + to] = key;
          idx_out[out + to] = payload_of(t);
        }
      }
      continue;
    }
    // Crowded bins.  From here on a thread holds the elements of its LDS slots.  Its number is made
    // opaque, or the compiler would keep this part's addresses in registers throughout.
    uint32_t ht = tid;
    asm volatile("" : "+v"(ht));
    uint32_t tmin = ~0u, tmax = 0;
#pragma unroll 1
    for (int r = 0; r < E; ++r) {
      const uint32_t i = (uint32_t)r * FT + ht;
      if (i >= gm) break;
      const uint64_t key = s_k[i];
      const uint32_t t = s_p[i];
      tmin = min(tmin, t);
      tmax = max(tmax, t);
      const uint32_t bin = bin_of(key, t);
      const uint32_t lo = s_bin.bin[bin], hi = bin_end(bin);
      if (hi - lo > BIN_MAX) {
        const uint64_t mid = s_k[(lo + hi) / 2];
        if (key != mid) atomicAdd(&s_side[bin], key < mid ? 1u : 1u << 16);
      }
    }
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      tmin = min(tmin, (uint32_t)__shfl_xor((int)tmin, off, WAVE));
      tmax = max(tmax, (uint32_t)__shfl_xor((int)tmax, off, WAVE));
    }
    if (lane_id() == 0) {
      atomicMin(&s_tmin, tmin);
      atomicMax(&s_tmax, tmax);
    }
    __syncthreads();
    tmin = uniform32(s_tmin);
    const uint32_t tspan = uniform32(s_tmax) - tmin;
    const uint32_t tbits = tspan ? 32u - (uint32_t)__clz((int)tspan) : 0u;
    // The place of an element with its bin's middle key, or ~0.
    auto place_of = [&](uint64_t key, uint32_t t, uint32_t bin, uint32_t lo, uint32_t hi) {
      if (hi - lo <= BIN_MAX || key != s_k[(lo + hi) / 2]) return ~0u;
      const uint32_t side = s_side[bin], less = side & 0xffffu;
      const uint32_t equal = hi - lo - less - (side >> 16);
      return lo + less + (uint32_t)(((uint64_t)(t - tmin) * equal) >> tbits);
    };
    auto count_place = [&](uint32_t q) {
      return (atomicAdd(&s_place[q / 2], 1u << (16 * (q & 1u))) >> (16 * (q & 1u))) & 0xffffu;
    };
    // at: an element's place (low half) and how many came to it before (high half), or ~0.
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const uint32_t i = (uint32_t)r * FT + ht;
      at[r] = ~0u;
      if (i < gm) {
        const uint64_t key = s_k[i];
        const uint32_t t = s_p[i];
        const uint32_t bin = bin_of(key, t);
        const uint32_t lo = s_bin.bin[bin], hi = bin_end(bin);
        const uint32_t side = hi - lo > BIN_MAX ? s_side[bin] : 0u;
        // Slots outside the middle key's part stand for one element each.
        if (hi - lo <= BIN_MAX || i < lo + (side & 0xffffu) || i >= hi - (side >> 16)) (void)count_place(i);
        const uint32_t q = place_of(key, t, bin, lo, hi);
        if (q != ~0u) {
          at[r] = q | (count_place(q) << 16);
        } else {
          const uint32_t to = rank_in(lo, hi, key, t);
          keys_out[out + to] = key;
          idx_out[out + to] = payload_of(t);
        }
      }
    }
    __syncthreads();
    // Exclusive scan of the places.
    uint32_t pw[WORDS], psum = 0;
#pragma unroll
    for (int q = 0; q < WORDS; ++q) {
      pw[q] = s_place[WORDS * ht + q];
      psum += (pw[q] & 0xffffu) + (pw[q] >> 16);
    }
    uint32_t pincl = psum;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      const uint32_t z = __shfl_up(pincl, off, WAVE);
      if (lane_id() >= off) pincl += z;
    }
    if (lane_id() == WAVE - 1) s_bin.w[wave] = pincl;
    __syncthreads();
    uint32_t prun = pincl - psum;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) prun += w < wave ? s_bin.w[w] : 0u;
#pragma unroll
    for (int q = 0; q < WORDS; ++q) {
      const uint32_t c = pw[q];
      s_place[WORDS * ht + q] = prun | ((prun + (c & 0xffffu)) << 16);
      prun += (c & 0xffffu) + (c >> 16);
    }
    // The ties of the middle keys' elements move to their places, within their bin's part.
#pragma unroll
    for (int r = 0; r < E; ++r) p[r] = at[r] != ~0u ? s_p[(uint32_t)r * FT + ht] : 0u;
    __syncthreads();
    auto prefix = [&](uint32_t q) { return (s_place[q / 2] >> (16 * (q & 1u))) & 0xffffu; };
#pragma unroll
    for (int r = 0; r < E; ++r)
      if (at[r] != ~0u) s_p[prefix(at[r] & 0xffffu) + (at[r] >> 16)] = p[r];
    __syncthreads();
    // Slot i still has its bin's key (or, where all keys are equal, tie), and in the middle key's
    // part one of its ties.
#pragma unroll 1
    for (int r = 0; r < E; ++r) {
      const uint32_t i = (uint32_t)r * FT + ht;
      if (i >= gm) break;
      const uint32_t t = s_p[i];
      const uint32_t bin = bin_of(s_k[i], t);
      const uint32_t lo = s_bin.bin[bin], hi = bin_end(bin);
      if (hi - lo <= BIN_MAX) continue;
      const uint32_t side = s_side[bin];
      if (i < lo + (side & 0xffffu) || i >= hi - (side >> 16)) continue;
      const uint64_t mid = s_k[(lo + hi) / 2];
      const uint32_t q = place_of(mid, t, bin, lo, hi);
      const uint32_t p0 = prefix(q), p1 = q + 1 < BUCKET_CAP ? prefix(q + 1) : gm;
      uint32_t to = p0;
      for (uint32_t j = p0; j < p1; ++j) to += s_p[j] < t ? 1u : 0u;
      keys_out[out + to] = mid;
      idx_out[out + to] = payload_of(t);
    }
  }
}

// ------------------------------------------------------------------ launcher
template <int E, int B>
static hipError_t sample_sort_shape(const uint64_t* keys, const uint8_t* ops, uint32_t n,
                                    uint64_t* tmp_keys, uint32_t* tmp_ties, uint64_t* keys_out,
                                    uint32_t* idx_out, const SampleControl& ctl, uint8_t* found,
                                    hipStream_t s) {
  constexpr uint32_t TILE = FT * E;
  static_assert(B <= (int)BUCKETS_MAX && B % 8 == 0, "bucket numbers are dealt to eight XCDs");
  const uint32_t tiles = (n + TILE - 1) / TILE;
  if (tiles > TILES_MAX) return hipErrorInvalidValue;
  constexpr int S = (int)PER_BUCKET * B;
  const SampleScratch sc = sample_scratch(ctl.words, B);
  // The raw samples lie where the sorted keys go.
  uint64_t* raw = S > 4096 ? keys_out : nullptr;
  if (raw) k_sample_fetch<S><<<S / 256, 256, 0, s>>>(keys, n, raw);
  k_sample_pick<S><<<S / FT, FT, 0, s>>>(keys, raw, n, sc, ctl.stall, ctl.barrier);
  k_sample_split<E, B><<<tiles, FT, 0, s>>>(keys, ops, n, sc, ctl.need, tmp_keys, tmp_ties, found);
  k_sample_bucket<<<B, FT, 0, s>>>(n, TILE, B, sc, tmp_keys, tmp_ties, keys_out, idx_out, ctl.need);
  return hipGetLastError();
}

// k_sample_bucket's shape is 1024 threads of four elements at every size: with two elements (half the
// LDS) or 512 threads a bucket that overflows, one in a hundred, comes to set the time (8 streamed
// batches of 2^21 ops 2665 µs with either, 2620-2690 with this; 2^19-op call 122-126 µs, with this 114).
size_t sample_sort_words(uint64_t n) {
  if (n < SAMPLE_SORT_MIN) return 0;
  return sample_words_of(n <= (1u << 19) ? 512u : n <= (1u << 20) ? 1024u : 2048u);
}

hipError_t sample_sort(const uint64_t* keys, const uint8_t* ops, uint32_t n, uint64_t* tmp_keys,
                       uint32_t* tmp_ties, uint64_t* keys_out, uint32_t* idx_out,
                       const SampleControl& ctl, uint8_t* found, hipStream_t s) {
  if (!sample_sorted(n)) return hipErrorInvalidValue;
  if (n <= (1u << 19))
    return sample_sort_shape<2, 512>(keys, ops, n, tmp_keys, tmp_ties, keys_out, idx_out, ctl, found, s);
  if (n <= (1u << 20))
    return sample_sort_shape<4, 1024>(keys, ops, n, tmp_keys, tmp_ties, keys_out, idx_out, ctl, found, s);
  if (n <= (1u << 21))
    return sample_sort_shape<8, 2048>(keys, ops, n, tmp_keys, tmp_ties, keys_out, idx_out, ctl, found, s);
  return sample_sort_shape<16, 2048>(keys, ops, n, tmp_keys, tmp_ties, keys_out, idx_out, ctl, found, s);
}

}  // namespace stm
