// Which of a step's items (sequences, experts) a workgroup belongs to, when item i has count(i) workgroups in a row.
#pragma once
#include "common.h"

namespace vgate {

// Inclusive sum over the lanes of a whole wave, on the VALU (rows of 16 shifted by 1, 2, 4, 8, then the last lanes of row 0 and 2 and
// of row 1 handed on): the six cross-lane trips through LDS of shuffles took 0.4 us at the head of a kernel of 11.
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// The item that holds number `want`, and its place in it (`local`); -1 past the last. Whole waves: a lane per item. Walking the items
// costs a trip to the scalar cache each, at the head of every workgroup (32 sequences: 3 us of a kernel of 8).
template <typename F>
__device__ __forceinline__ int locate_item(int n, int want, int& local, F count) {
  const int lane = threadIdx.x & 63;
  int base = 0;
  for (int i0 = 0; i0 < n; i0 += 64) {
    const int c = i0 + lane < n ? count(i0 + lane) : 0;
    const int end = wave_scan(c);
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
  return __builtin_amdgcn_readlane(wave_scan(c), 63);
}

}  // namespace vgate
