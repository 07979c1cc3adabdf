// What the recurrences that take a portion in chunks of CN tokens share (gated_delta.hip, delta_rule.hip): where a chunk
// lies, sums over lanes, packed lower triangles and their products with a column kept in registers.
#pragma once
#include "locate.h"

namespace vgate {
namespace {

constexpr int CN = 32;   // tokens of a chunk

template <int CTRL>
__device__ __forceinline__ float row_rot(float v) {  // a rotation inside each row of 16 lanes (DPP), on the VALU
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// sum over the KG lanes that share lane % (64 / KG)
template <int KG>
__device__ __forceinline__ float key_sum(float v) {
  if (KG >= 32) v += row_rot<0x122>(v);   // lanes 2 apart
  if (KG >= 16) v += row_rot<0x124>(v);   // 4
  v += row_rot<0x128>(v);                 // 8
  v += xor16(v);
  v += xor32(v);
  return v;
}

// chunks of C tokens of sequence i (sequences without a slot, or of at most `lim` tokens, have none)
template <int C>
__device__ __forceinline__ int chunks_of(const int32_t* state_slots, int lim, int i, int a, int b) {
  return (state_slots[i] < 0 || b - a <= lim) ? 0 : (b - a + C - 1) / C;
}

// chunk `bx` of a step: its sequence and token range (chunks are numbered sequence by sequence)
template <int C = CN>
__device__ __forceinline__ bool locate_chunk(const int32_t* query_start, const int32_t* state_slots, int S, int lim, int bx, int& s,
                                             int& t0, int& t1) {
  int local;
  s = locate_item(S, bx, local, [&](int i) { return chunks_of<C>(state_slots, lim, i, query_start[i], query_start[i + 1]); });
  if (s < 0) return false;
  t0 = query_start[s] + local * C;
  t1 = min(query_start[s + 1], t0 + C);
  return true;
}

// number of the first chunk of sequence s
template <int C = CN>
__device__ __forceinline__ int first_chunk(const int32_t* query_start, const int32_t* state_slots, int lim, int s) {
  return count_items(s, [&](int i) { return chunks_of<C>(state_slots, lim, i, query_start[i], query_start[i + 1]); });
}

// sum over j < n (a constant after unrolling) of row[j] x[j]; the row is read in 16-B pieces
__device__ __forceinline__ float row_dot(const float* row, const float (&x)[CN], int n) {
  float a = 0.f, b = 0.f;   // (two chains)
#pragma unroll
  for (int j0 = 0; j0 < CN; j0 += 4)
    if (j0 < n) {
      const float4 v = *reinterpret_cast<const float4*>(row + j0);
      a = fmaf(v.x, x[j0], a);
      if (j0 + 1 < n) b = fmaf(v.y, x[j0 + 1], b);
      if (j0 + 2 < n) a = fmaf(v.z, x[j0 + 2], a);
      if (j0 + 3 < n) b = fmaf(v.w, x[j0 + 3], b);
    }
  return a + b;
}

// first float of row i of a packed lower triangle whose row i has i entries, padded to whole 16-B pieces (row i of one with
// the diagonal: tri(i + 1))
__host__ __device__ constexpr int tri(int i) {
  const int n = i > 0 ? i - 1 : 0, g = n / 4;
  return i > 0 ? 4 * (2 * g * (g + 1) + (n - 4 * g) * (g + 1)) : 0;
}

__device__ __forceinline__ f32x4 ld4(const float* p) {
  const float4 v = *reinterpret_cast<const float4*>(p);
  return f32x4{v.x, v.y, v.z, v.w};
}

// Where element (row, k) of an MFMA operand lies in a record: [16-row tile][16-k tile of kt][lane = (k quad, row)][4 k], so that a wave's
// load of a 16-B piece per lane is one KiB in a row. (With rows in a row, 64 lanes touched 16 lines of which they took 64 B: the address
// path bound the chunk scans. 2048 tokens, 8 heads of 128, delta rule 154 -> 112 us, gated 82 -> 60.)
__device__ __forceinline__ int frag(int row, int k, int kt) {
  return (((row >> 4) * kt + (k >> 4)) * 64 + ((k >> 2) & 3) * 16 + (row & 15)) * 4 + (k & 3);
}
__host__ __device__ constexpr int whole16(int n) { return (n + 15) / 16 * 16; }

// Rows row0 .. row0 + 3 of column c, one column per lane of whole quads (c % 4 = lane % 4), into a record: turned so that a lane stores four
// columns of one row, a 16-B piece.
__device__ __forceinline__ void put_rows4(float* base, int row0, int c, int kt, f32x4 v) {
  const bool odd = c & 1, high = c & 2;
  const float x0 = row_rot<0xB1>(odd ? v[0] : v[1]), x1 = row_rot<0xB1>(odd ? v[2] : v[3]);   // (quad_perm [1, 0, 3, 2])
  v = odd ? f32x4{x0, v[1], x1, v[3]} : f32x4{v[0], x0, v[2], x1};
  const float y0 = row_rot<0x4E>(high ? v[0] : v[2]), y1 = row_rot<0x4E>(high ? v[1] : v[3]);   // ([2, 3, 0, 1])
  v = high ? f32x4{y0, y1, v[2], v[3]} : f32x4{v[0], v[1], y0, y1};
  *reinterpret_cast<f32x4*>(base + frag(row0 + (c & 3), c & ~3, kt)) = v;
}

// sum over the 32 lanes of a half wave, in all of them
__device__ __forceinline__ float half_sum(float v) {
  v += row_rot<0x128>(v);
  v += row_rot<0x124>(v);
  v += row_rot<0x122>(v);
  v += row_rot<0x121>(v);
  return v + xor16(v);
}

}  // namespace
}  // namespace vgate
