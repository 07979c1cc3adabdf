// Which of a step's items (sequences, experts) a workgroup belongs to, when item i has count(i) workgroups in a row.
#pragma once
#include "common.h"

namespace vgate {

// The item that holds number `want`, and its place in it (`local`); -1 past the last. Whole waves: a lane per item. Walking the items
// costs a trip to the scalar cache each, at the head of every workgroup (32 sequences: 3 us of a kernel of 8).
template <typename F>
__device__ __forceinline__ int locate_item(int n, int want, int& local, F count) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int c = i0 + lane < n ? count(i0 + lane) : 0;
    int end = c;   // inclusive sum over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(end, o, 64);
      if (lane >= o) end += v;
    }
    const unsigned long long hit = __ballot(want >= base + end - c && want < base + end);
    if (hit != 0) {
      const int l = __ffsll(hit) - 1;
      local = want - base - __builtin_amdgcn_readlane(end - c, l);
      return i0 + l;
    }
    base += __builtin_amdgcn_readlane(end, 63);
  }
  return -1;
}

// sum of count(i) over i < n (whole waves)
template <typename F>
__device__ __forceinline__ int count_items(int n, F count) {
  int c = 0;
  for (int i = threadIdx.x & 63; i < n; i += 64) c += count(i);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  return __builtin_amdgcn_readfirstlane(c);
}

}  // namespace vgate
