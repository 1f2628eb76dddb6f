// stm_binsort.hpp — sort of the elements of one workgroup in LDS, for the sample sorts of small
// batches (stm_front.hip) and large ones (stm_sample.hip).
#pragma once
#include "stm_common.hpp"
#include "stm_internal.hpp"

namespace stm {

constexpr int FT = 1024;  // threads of every workgroup of the sample sorts
constexpr int FW = FT / WAVE;

// An element is (key, tie): the tie is the input position with the op code below it, so ties are
// distinct and the order is the stable order.  Padding is (KEY_EMPTY, ~0), above every element.
STM_DEV bool elem_less(uint64_t ka, uint32_t pa, uint64_t kb, uint32_t pb) {
  return ka < kb || (ka == kb && pa < pb);
}

// Value of the lane whose number differs in bit x (a power of two below 64).  Written as a
// switch over literals, which unrolled callers fold: the lane swaps inside a quad are a register
// move, those up to 16 lanes need no address.
STM_DEV uint32_t lane_xor(uint32_t v, int x) {
  switch (x) {
    case 1: return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, true);
    case 2: return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, true);
    case 4: return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (4 << 10) | 0x1F);
    case 8: return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (8 << 10) | 0x1F);
    case 16: return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (16 << 10) | 0x1F);
    default: return (uint32_t)__shfl_xor((int)v, 32, WAVE);
  }
}

// Bitonic sort of N elements held E per thread by the first N / E threads: element tid * E + r in
// k[r], p[r] (any order on entry).  A step of distance below E stays in the thread, below 64 * E
// in the wavefront; the others (10 of 66 at N = 2048) go through LDS (N elements of s_k, s_p).
// Every thread of the workgroup calls it.
template <int N, int E>
STM_DEV void block_sort(uint64_t (&k)[E], uint32_t (&p)[E], uint64_t* s_k, uint32_t* s_p) {
  constexpr int NT = N / E;
  static_assert(NT % WAVE == 0 && NT <= FT, "whole wavefronts of the workgroup");
  const uint32_t tid = threadIdx.x;
  const bool act = tid < (uint32_t)NT;
#pragma unroll
  for (int size = 2; size <= N; size <<= 1) {
#pragma unroll
    for (int d = size >> 1; d > 0; d >>= 1) {
      if (d < E) {
#pragma unroll
        for (int r = 0; r < E; ++r) {
          if (r & d) continue;
          const bool up = ((tid * E + r) & (uint32_t)size) == 0;
          const bool swap = elem_less(k[r ^ d], p[r ^ d], k[r], p[r]) == up;
          const uint64_t ka = k[r], kb = k[r ^ d];
          const uint32_t pa = p[r], pb = p[r ^ d];
          k[r] = swap ? kb : ka;
          p[r] = swap ? pb : pa;
          k[r ^ d] = swap ? ka : kb;
          p[r ^ d] = swap ? pa : pb;
        }
      } else {
        const bool through_lds = d >= WAVE * E;
        if (through_lds) {
          __syncthreads();
          if (act) {
#pragma unroll
            for (int r = 0; r < E; ++r) {
              s_k[r * NT + tid] = k[r];
              s_p[r * NT + tid] = p[r];
            }
          }
          __syncthreads();
        }
        if (act) {
          const bool up = ((tid * E) & (uint32_t)size) == 0;
          const bool lower = ((tid * E) & (uint32_t)d) == 0;
          const bool keep_min = up == lower;
#pragma unroll
          for (int r = 0; r < E; ++r) {
            uint64_t pk;
            uint32_t pp;
            if (through_lds) {
              pk = s_k[r * NT + (tid ^ (uint32_t)(d / E))];
              pp = s_p[r * NT + (tid ^ (uint32_t)(d / E))];
            } else {
              const uint32_t lo = lane_xor((uint32_t)k[r], d / E);
              const uint32_t hi = lane_xor((uint32_t)(k[r] >> 32), d / E);
              pk = ((uint64_t)hi << 32) | lo;
              pp = lane_xor(p[r], d / E);
            }
            const bool take = elem_less(pk, pp, k[r], p[r]) == keep_min;
            k[r] = take ? pk : k[r];
            p[r] = take ? pp : p[r];
          }
        }
      }
    }
  }
}

// LDS of bin_sort beside the elements.
constexpr uint32_t BIN_BITS = 11;
constexpr uint32_t BINS = 1u << BIN_BITS;
constexpr uint32_t BIN_MAX = 32;  // a bin with more elements sends the block to the comparison sort
struct BinShared {
  uint32_t bin[BINS];
  uint64_t mn, mx;  // least and greatest key
  uint32_t heavy;
  uint32_t w[FW];
};

// Before the first barrier ahead of bin_sort.
template <int NT>
STM_DEV void bin_sort_open(BinShared& sh) {
#pragma unroll
  for (uint32_t q = threadIdx.x; q < BINS; q += NT) sh.bin[q] = 0;
  if (threadIdx.x == 0) {
    sh.mn = KEY_EMPTY;
    sh.mx = 0;
    sh.heavy = 0;
  }
}

// The block's m <= NT * E elements, element r * NT + tid in k[r], p[r], into sorted order in s_k, s_p.
// They are counted into BINS bins by the leading bits of their key within the block's range (of
// their tie where all keys are equal), placed by bin and ranked among the few elements of their
// bin.  Keys that crowd a bin (a hot key, tight clusters) are sorted by comparison.
// The comparison sort is bound by its arithmetic: 55 steps of some 14 instructions per element at
// 1024 elements, where a lane of this one executes about 100.  Comparison sort / this, µs:
// k_front_small of 1000 ops 9.1 / 7.2, k_front_bucket of 40001 ops 11.2 / 7.7, k_front_split of 131075
// ops (2048 samples) 19.4 / 16.8; with crowded bins (Zipf inserts, 2^14 ops) no difference.
// Every thread of the workgroup calls it, after bin_sort_open and a barrier.
template <int NT, int E>
STM_DEV void bin_sort(uint32_t m, uint64_t (&k)[E], uint32_t (&p)[E], uint64_t* s_k, uint32_t* s_p,
                      BinShared& sh) {
  const uint32_t tid = threadIdx.x;
  const uint32_t wave = tid / WAVE;
  uint64_t mn = KEY_EMPTY, mx = 0;
#pragma unroll
  for (int r = 0; r < E; ++r) {
    if ((uint32_t)r * NT + tid < m) {
      mn = k[r] < mn ? k[r] : mn;
      mx = k[r] > mx ? k[r] : mx;
    }
  }
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const uint64_t a = ((uint64_t)lane_xor((uint32_t)(mn >> 32), off) << 32) | lane_xor((uint32_t)mn, off);
    const uint64_t b = ((uint64_t)lane_xor((uint32_t)(mx >> 32), off) << 32) | lane_xor((uint32_t)mx, off);
    mn = a < mn ? a : mn;
    mx = b > mx ? b : mx;
  }
  if (lane_id() == 0 && wave * WAVE < m) {
    atomicMin((unsigned long long*)&sh.mn, (unsigned long long)mn);
    atomicMax((unsigned long long*)&sh.mx, (unsigned long long)mx);
  }
  __syncthreads();
  mn = sh.mn;
  mx = sh.mx;
  const bool same = mn == mx;
  const uint32_t len = same ? 32u : mx ? 64u - (uint32_t)__clzll((long long)(mx - mn)) : 0u;
  const uint64_t base = same ? 0ull : mn;
  const uint32_t shift = len > BIN_BITS ? len - BIN_BITS : 0u;
  uint32_t bin[E], at[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    bin[r] = 0;
    at[r] = 0;
    if ((uint32_t)r * NT + tid < m) {
      bin[r] = (uint32_t)(((same ? (uint64_t)p[r] : k[r]) - base) >> shift);
      at[r] = atomicAdd(&sh.bin[bin[r]], 1u);
      if (at[r] >= BIN_MAX) sh.heavy = 1;
    }
  }
  __syncthreads();
  if (sh.heavy) {
#pragma unroll
    for (int r = 0; r < E; ++r) {
      const bool v = (uint32_t)r * NT + tid < m;
      k[r] = v ? k[r] : KEY_EMPTY;
      p[r] = v ? p[r] : ~0u;
    }
    block_sort<NT * E, E>(k, p, s_k, s_p);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < E; ++r) {
      s_k[tid * E + r] = k[r];
      s_p[tid * E + r] = p[r];
    }
    __syncthreads();
    return;
  }
  // Exclusive scan of the bins, PER per thread.
  constexpr uint32_t PER = BINS / NT;
  uint32_t c[PER], sum = 0;
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    c[q] = sh.bin[tid * PER + q];
    sum += c[q];
  }
  uint32_t x = sum;
#pragma unroll
  for (int off = 1; off < WAVE; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, WAVE);
    if (lane_id() >= off) x += y;
  }
  if (lane_id() == WAVE - 1) sh.w[wave] = x;
  __syncthreads();
  uint32_t run = x - sum;
#pragma unroll
  for (int w = 0; w < NT / WAVE; ++w) run += (uint32_t)w < wave ? sh.w[w] : 0u;
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    sh.bin[tid * PER + q] = run;
    run += c[q];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    if ((uint32_t)r * NT + tid < m) {
      at[r] += sh.bin[bin[r]];
      s_k[at[r]] = k[r];
      s_p[at[r]] = p[r];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    if ((uint32_t)r * NT + tid < m) {
      const uint32_t lo = sh.bin[bin[r]];
      const uint32_t hi = bin[r] + 1 < BINS ? sh.bin[bin[r] + 1] : m;
      at[r] = lo;
      if (hi - lo > 1)
        for (uint32_t j = lo; j < hi; ++j) at[r] += elem_less(s_k[j], s_p[j], k[r], p[r]) ? 1u : 0u;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < E; ++r) {
    if ((uint32_t)r * NT + tid < m) {
      s_k[at[r]] = k[r];
      s_p[at[r]] = p[r];
    }
  }
  __syncthreads();
}

// The tie of input position i: the position, then the op code (codes above 3 are GETs).
STM_DEV uint32_t tie_of(uint32_t i, uint32_t op) { return (i << 2) | (op > 3u ? 1u : op); }
STM_DEV uint32_t payload_of(uint32_t tie) { return (tie >> 2) | (tie << POS_BITS); }

// Where within its stretch of the input a sample is drawn: lowbias32, the 32-bit integer hash that
// Chris Wellons published with his hash-prospector (public domain).
STM_DEV uint32_t hash32(uint32_t x) {
  x = (x ^ (x >> 16)) * 0x7feb352du;
  x = (x ^ (x >> 15)) * 0x846ca68bu;
  return x ^ (x >> 16);
}

}  // namespace stm
