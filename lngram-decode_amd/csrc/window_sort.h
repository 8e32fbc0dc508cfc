// Counting sort of one route's window keys by a block of 1024 threads (table and lookup gradients).
#pragma once

#include "common.h"

namespace lng {

constexpr uint32_t WIN_DEAD = 0xFFFF;  // key of a position without a gradient (rows per route <= 2^13)

// keys: the route's `kstride` uint16 keys, a multiple of 64 (WIN_DEAD past the last position); S rows
// (a power of two); start[S + 1] gets the first list index of each row, perm the positions in row
// order (the order within a row varies), each shifted left by `pack` with its key below when pack > 0.
// cnt: S + 16 words of LDS.  Keys are read 8 a thread.
__device__ __forceinline__ void sort_windows(const uint16_t* __restrict__ keys, int64_t kstride, int S, int pack,
                                             uint32_t* __restrict__ start, uint32_t* __restrict__ perm,
                                             uint32_t* cnt) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t* wsum = cnt + S;
  const u32x4* kr = reinterpret_cast<const u32x4*>(keys);
  const int64_t nv = kstride / 8;
  for (int i = tid; i < S; i += 1024) cnt[i] = 0;
  __syncthreads();
  for (int64_t i = tid; i < nv; i += 1024) {
    const u32x4 q = kr[i];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t key = (q[j >> 1] >> (16 * (j & 1))) & 0xFFFF;
      if (key != WIN_DEAD) atomicAdd(&cnt[key], 1u);
    }
  }
  __syncthreads();
  // exclusive scan of the counters: a thread's S / 1024 consecutive ones, then the threads' totals
  const int per = S > 1024 ? S / 1024 : 1;
  const int c0 = tid * per;
  uint32_t sum = 0;
  if (c0 < S)
    for (int i = 0; i < per; ++i) sum += cnt[c0 + i];
  uint32_t inc = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t o = __shfl_up(inc, d);
    if (lane >= d) inc += o;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  uint32_t base = inc - sum;
  for (int i = 0; i < wave; ++i) base += wsum[i];
  if (c0 < S) {
    for (int i = 0; i < per; ++i) {
      const uint32_t c = cnt[c0 + i];
      cnt[c0 + i] = base;
      start[c0 + i] = base;
      base += c;
    }
    if (c0 + per == S) start[S] = base;
  }
  __syncthreads();
  for (int64_t i = tid; i < nv; i += 1024) {
    const u32x4 q = kr[i];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t key = (q[j >> 1] >> (16 * (j & 1))) & 0xFFFF;
      if (key != WIN_DEAD)
        perm[atomicAdd(&cnt[key], 1u)] = (static_cast<uint32_t>(i * 8 + j) << pack) | (pack ? key : 0u);
    }
  }
}

}  // namespace lng
