// Rows of a bf16 matrix staged in LDS by DMA so that both sides are fast: whole 128-B lines from memory, MFMA fragments free of bank
// conflicts out of LDS (gemm_prefill.hip, gemm_prompt.h, gemm_prompt_q4.hip, gemm_mid.hip, latent_attn.hip).
#pragma once
#include "common.h"

namespace vgate {

// ---- x in LDS: a 16-row x 64-k tile is two 1 KiB pieces of 8 rows ----
// Eight consecutive lanes of the DMA fetch one row's whole 128-B line. (Gathering MFMA fragments directly, 64 lanes on 16 rows of
// 64 B each, kept the CU's address path busy four times as long and bounded every tile shape at 20 to 22 B per clock and CU: 1536 x
// 8960 at 2048 rows as 128 x 128 tiles 115 -> 88 us, 4096 x 4096 as 256 x 128 92 -> 73, 28672 x 4096 as 256 x 128 545 -> 476.) LDS-DMA
// writes lane-linear, so the 16-B chunks of a row are permuted at the source: chunk c of row r lies at c ^ x_swz(r), which spreads the
// 16 rows of a fragment read over all banks (SQ_LDS_BANK_CONFLICT 0).
__device__ __forceinline__ int x_swz(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int x_piece_row(int tile_row0, int half, int lane, int M) {
  const int row = tile_row0 + 8 * half + (lane >> 3);
  return row < M ? row : M - 1;  // rows past M repeat row M - 1 (never stored)
}
__device__ __forceinline__ int x_piece_col(int half, int lane) { return ((lane & 7) ^ x_swz(8 * half + (lane >> 3))) * 8; }
__device__ __forceinline__ int x_frag_off(int ks, int lane) {
  const int r = lane & 15;
  return r * 128 + (((4 * ks + (lane >> 4)) ^ x_swz(r)) << 4);
}

// LDS-DMA through a buffer descriptor: 16 B per lane from base + voff + soff to lds + 16 lane (inline asm and vmcnt by the caller, as
// glds16; no 64-bit address per piece: a wave that issues alone on its SIMD has no slots for those)
__device__ __forceinline__ void blds16(u32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\ts_mov_b32 m0, %0"
               : "=&s"(keep) : "v"(voff), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
}
// N of them off one setting of M0, the i-th 1 KiB i further in memory and in LDS (the instruction's offset counts in both)
template <int N>
__device__ __forceinline__ void blds16_run(u32x4 rsrc, const uint32_t (&voff)[N], uint32_t soff, uint32_t lds) {
  static_assert(N >= 1 && N <= 4, "the offset has 12 bits");
  unsigned keep;
  if constexpr (N == 1)
    blds16(rsrc, voff[0], soff, lds);
  else if constexpr (N == 3)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %6\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %4, %5 offen lds\n\t"
                 "buffer_load_dwordx4 %2, %4, %5 offen offset:1024 lds\n\tbuffer_load_dwordx4 %3, %4, %5 offen offset:2048 lds\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
  else if constexpr (N == 2)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %5\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %3, %4 offen lds\n\t"
                 "buffer_load_dwordx4 %2, %3, %4 offen offset:1024 lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(voff[0]), "v"(voff[1]), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %7\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %5, %6 offen lds\n\t"
                 "buffer_load_dwordx4 %2, %5, %6 offen offset:1024 lds\n\tbuffer_load_dwordx4 %3, %5, %6 offen offset:2048 lds\n\t"
                 "buffer_load_dwordx4 %4, %5, %6 offen offset:3072 lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep) : "v"(voff[0]), "v"(voff[1]), "v"(voff[2]), "v"(voff[3]), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
}
__device__ __forceinline__ u32x4 rsrc_words(const void* base) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)), 0x7fffffffu, 0x00020000u};
}

// acc += W(A) . X(B) on an accumulator that stays in its AGPRs: up to 256 of them are the whole file, and with the builtin (whose result is
// another register than its addend) the allocator shuffles them through VGPRs all the way. The compiler does not see an MFMA here, so the
// waits that it would put around one are the caller's: operands come from LDS (waited for as any asm input) or, written by the VALU, with
// two wait states between; before the accumulators are read, the last MFMA is given its 16 cycles and more.
__device__ __forceinline__ void mfma_acc(f32x4& acc, const uint4& w, const uint4& x) {
  asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(as_bf16x8(w)), "v"(as_bf16x8(x)));
}

// eight scores in log2 units become softmax weights 2^(v - ms), and their sum. (The bare instruction gives zero below 2^-126, where a
// large value may still count: a wave that meets such a weight takes exp2f(), five instructions more each.)
__device__ __forceinline__ float weights8(float (&v)[8], float ms) {
  float least = v[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) least = fminf(least, v[e]);
  float sum = 0.f;
  if (__any(least - ms < -126.f)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = exp2f(v[e] - ms);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = __builtin_amdgcn_exp2f(v[e] - ms);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) sum += v[e];
  return sum;
}

}  // namespace vgate
