// The norm of one row by a workgroup of 256 threads: y = (x - mean) / sqrt(mean((x - mean)^2) + eps), the mean 0 unless `center`.
// Thread t holds columns t, t + 256, ..: the first NI of them in registers, what lies beyond is asked for again. Every kernel that makes
// a normed row sums in this order, so which kernel makes it does not change its bits.
#pragma once
#include "common.h"

namespace vgate {

// v[i]: column threadIdx.x + 256 i; rest(c): a column from 256 NI on; put(c, i, y): i the register's index, -1 beyond. `red`: 16 floats
// of LDS. All 256 threads.
template <int NI, typename Rest, typename Put>
__device__ __forceinline__ void norm_row(const float (&v)[NI], int n, float eps, int center, float* red, Rest rest, Put put) {
  const int tid = threadIdx.x;
  float mean = 0.f;
  if (center) {  // (uniform)
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i)
      if (tid + 256 * i < n) s += v[i];
    for (int c = tid + 256 * NI; c < n; c += 256) s += rest(c);
    mean = block_reduce_sum(s, red) / (float)n;
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (tid + 256 * i < n) {
      const float d = v[i] - mean;
      ss = fmaf(d, d, ss);
    }
  for (int c = tid + 256 * NI; c < n; c += 256) {
    const float d = rest(c) - mean;
    ss = fmaf(d, d, ss);
  }
  const float inv = 1.f / sqrtf(block_reduce_sum(ss, red) / (float)n + eps);
#pragma unroll
  for (int i = 0; i < NI; ++i)
    if (tid + 256 * i < n) put(tid + 256 * i, i, (v[i] - mean) * inv);
  for (int c = tid + 256 * NI; c < n; c += 256) put(c, -1, (rest(c) - mean) * inv);
}

// columns c of a bf16 or fp32 row, thread by thread, all loads together (past n: the last column's)
template <int NI>
__device__ __forceinline__ void load_row(const void* x, int64_t ro, int f32, int n, float (&v)[NI]) {
  if (f32) {  // (uniform)
#pragma unroll
    for (int i = 0; i < NI; ++i) v[i] = reinterpret_cast<const float*>(x)[ro + min((int)threadIdx.x + 256 * i, n - 1)];
  } else {
#pragma unroll
    for (int i = 0; i < NI; ++i) v[i] = bf2f(reinterpret_cast<const bf16_t*>(x)[ro + min((int)threadIdx.x + 256 * i, n - 1)]);
  }
}

}  // namespace vgate
