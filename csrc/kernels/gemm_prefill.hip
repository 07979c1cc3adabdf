// LDS-tiled MFMA GEMM for prefill / long steps (M >= 128) on gfx950 — the hand-written
// replacement of the hipBLASLt path, on the SAME fragment-packed weights the decode kernels
// stream (no second plain copy of any weight is kept).
//
//   out[m][n] = epilogue( rowscale(m) * sum_k x[m][k] * W[n][k] )
//
// Both operands are staged global -> LDS by LDS-DMA (global_load_lds_dwordx4, 1 KiB per wave
// instruction) into a 2-deep ring, BK = 64 (two 32-deep MFMA k-steps per stage):
//   * W: the packed layout Wp[nt][kt][lane][8] IS the MFMA A-fragment order, so one 1 KiB
//     piece (one 16-column tile x one k-step) lands lane-linear and every wave reads its
//     fragments back with conflict-free ds_read_b128 (lane l at +16 l) — no swizzle needed;
//   * x: each 1 KiB piece is 8 rows x 64 k, eight consecutive lanes to a 128-B line (x_piece_row).
// Pipeline (cdna_hip_programming.md §5 'glds vs register staging', first row): the stage t+1
// DMA is issued before stage t's ds_reads + MFMAs, one vmcnt(0) + barrier per stage.
// Block tile BM x BN over 4 waves (2 x 2), wave tile (BM/2) x (BN/2) in 16x16x32 bf16 MFMAs,
// orientation D = W(A) . X(B): lane holds D[n = 4(l>>4)+i][m = l&15], so the epilogues of the
// decode kernels (gemm_epilogue.h: bias, residual, SiLU*mul pairs, QKV RoPE + KV write) are
// reused unchanged. The RMSNorm in front of qkv / gate_up runs as the deferred row scale
// (gamma folded into W at load time): x^2 is accumulated from the B fragments the MFMAs read.
// Grid: 1-D, XCD-aware bijective remap, m-blocks fastest so the blocks that share a weight
// column panel run back to back on one XCD (one HBM read of the panel per XCD L2).
#include <cstdlib>
#include <stdexcept>

#include "gemm_prompt.h"

namespace vgate {

template <int BM, int BN, int EPI, int NORM, int NTB>
__global__ __launch_bounds__(256, 2) void gemm_prefill_kernel(GemmParams p) {
  static_assert(BM % 32 == 0 && BN % 32 == 0, "2 x 2 waves of 16-multiple tiles");
  constexpr int KS = 2;                      // 32-deep k-steps per stage (BK = 64)
  constexpr int WTN = BN / 16, XTM = BM / 16;  // 16-wide tiles per block
  constexpr int NT = WTN / 2, MT = XTM / 2;    // per wave
  constexpr int PIECES = (WTN + XTM) * KS;     // 1 KiB pieces per stage
  static_assert(PIECES % 4 == 0, "pieces split evenly over 4 waves");
  constexpr int PPW = PIECES / 4;              // per wave
  constexpr int STAGE = PIECES * 1024;
  static_assert(NT % NTB == 0, "epilogue tile groups");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TLScope tl_scope(p.dbg_ts);
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const int KT = p.K >> 5;
  const int nk_all = p.K >> 6;  // stages (K % 64 == 0, host-checked)
  // split-K (small tile grids): blockIdx.y = K slice; partials go to the reduce kernel
  const int z = blockIdx.y, nz = gridDim.y;
  const int kst0 = (nk_all * z) / nz, nk = (nk_all * (z + 1)) / nz - kst0;
  // XCD-aware logical block id (bijective for any grid size), then m fastest
  const int mblocks = (p.M + BM - 1) / BM;
  const int nwg = gridDim.x, orig = blockIdx.x, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int wgid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  const int m0 = (wgid % mblocks) * BM;
  const int nt_blk = (wgid / mblocks) * WTN;  // first 16-column tile of the block
  // this wave's DMA pieces: piece f < WTN*KS is W tile f / KS at k-step f % KS, else x
  // m-tile (f - WTN*KS) / KS. Source addresses per lane, advanced by one stage per iteration.
  const char* src[PPW];
  int step[PPW];  // bytes per stage
#pragma unroll
  for (int i = 0; i < PPW; ++i) {
    const int f = wid * PPW + i;
    if (f < WTN * KS) {
      const int nt = nt_blk + f / KS, ks = f % KS;
      src[i] = reinterpret_cast<const char*>(p.wp) + (((size_t)nt * KT + 2 * kst0 + ks) * 64 + lane) * 16;
      step[i] = KS * 1024;
    } else {
      const int g = f - WTN * KS;
      const int row = x_piece_row(m0 + (g >> 1) * 16, g & 1, lane, p.M);
      src[i] = reinterpret_cast<const char*>(p.x + (size_t)row * p.lda + kst0 * 64 + x_piece_col(g & 1, lane));
      step[i] = 64 * 2;
    }
  }
  const uint32_t lds0 = lds_addr_of(smem);
  const int xo[2] = {x_frag_off(0, lane), x_frag_off(1, lane)};
  auto issue = [&](int stage, int buf) {
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
      const int f = wid * PPW + i;  // wave-uniform LDS destination (M0): lane l lands at +16 l
      glds16(src[i] + (size_t)stage * step[i], __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + f * 1024));
    }
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[MT];
#pragma unroll
  for (int b = 0; b < MT; ++b) ss[b] = 0.f;

  issue(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int t = 0; t < nk; ++t) {
    const int buf = t & 1;
    if (t + 1 < nk) issue(t + 1, buf ^ 1);
    const char* sb = smem + buf * STAGE;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 wa[NT], xb[MT];
#pragma unroll
      for (int a = 0; a < NT; ++a)
        wa[a] = *reinterpret_cast<const uint4*>(sb + ((wn * NT + a) * KS + ks) * 1024 + lane * 16);
#pragma unroll
      for (int b = 0; b < MT; ++b)
        xb[b] = *reinterpret_cast<const uint4*>(sb + (WTN + wm * MT + b) * 2048 + xo[ks]);
      if constexpr (NORM == 2) {
#pragma unroll
        for (int b = 0; b < MT; ++b) {
          ss[b] = sumsq8(xb[b], ss[b]);
        }
      }
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = mfma16(as_bf16x8(wa[a]), as_bf16x8(xb[b]), acc[a][b]);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  if (nz > 1) {
    // fp32 partial of this K slice -> slabs [z][M][N] (row-major, the lane's 4 columns as one
    // 16-B store) and its rows' partial sums of squares -> [z][M] after the tiles; the reduce
    // kernel sums the slices in a fixed order (bit-reproducible) and runs the epilogue
    float* part = p.slabs + (size_t)z * p.M * p.N;
    float* ssq = p.slabs + (size_t)nz * p.M * p.N + (size_t)z * p.M;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int m = m0 + wm * (BM / 2) + b * 16 + (lane & 15);
      if constexpr (NORM == 2) {
        float s2 = ss[b];
        s2 += xor16(s2);
        s2 += xor32(s2);
        if (wn == 0 && lane < 16 && m < p.M) ssq[m] = s2;
      }
      if (m < p.M) {
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          const int n = (nt_blk + wn * NT + a) * 16 + 4 * (lane >> 4);
          __builtin_nontemporal_store(acc[a][b], reinterpret_cast<f32x4*>(part + (size_t)m * p.N + n));
        }
      }
    }
    return;
  }
  // epilogue straight from the accumulators: row m = m0 + wm*(BM/2) + 16 b + (l & 15)
#pragma unroll
  for (int b = 0; b < MT; ++b) {
    const int m = m0 + wm * (BM / 2) + b * 16 + (lane & 15);
    float sc = 1.f;
    if constexpr (NORM == 2) {
      float s2 = ss[b];
      s2 += xor16(s2);
      s2 += xor32(s2);
      sc = rsqrtf(s2 / (float)p.K + p.eps);
    }
#pragma unroll
    for (int a = 0; a < NT; a += NTB) {
      f32x4 v[NTB];
#pragma unroll
      for (int j = 0; j < NTB; ++j) v[j] = acc[a + j][b] * sc;
      epilogue<NTB, EPI, false>(p, v, m, nt_blk + wn * NT + a, 4 * (lane >> 4), EpiPre<NTB>{}, m < p.M);
    }
  }
}

// ---- v2: deeper pipeline, bigger block tile ----
// Same operand staging (LDS-DMA of fragment-major 1 KiB pieces, conflict-free ds_read_b128),
// epilogues and split-K contract as gemm_prefill_kernel, but
//   * an NS-deep stage ring: stage t + NS - 1 is issued before stage t is consumed, with ONE
//     counted vmcnt wait + s_barrier per stage (no vmcnt(0): the NS-2 younger stages stay in
//     flight). The 2-deep ring waited for the stage it had just issued every 64 k, so each
//     stage paid a full L2 / HBM round trip (~0.5-1 us) against ~0.4 us of MFMA work;
//   * WM x WN waves (8: 512 threads) on a BM x BN = 256 x 128 tile, wave tile 64 x 64: twice the
//     MFMA work per staged byte of the 128 x 128 tile and one block per CU (144 KiB ring).
// Past the last stage the ring keeps issuing (clamped duplicate loads into buffers that are never
// read again), so every wait count is a compile-time constant.
// SCHED (k-loop schedule): 0 = the stage's DMA issued before its reads + MFMAs; 1 = + MFMAs at raised
// wave priority (s_setprio 1: the MFMA-issuing wave wins the SIMD's arbitration over the other wave's
// LDS reads / DMA issue); 2 = 1 + the stage's DMA issue split in two, half in front of each k-step
template <int BM, int BN, int WM, int WN, int NS, int EPI, int NORM, int NTB, int SCHED = 0, int KS = 2>
__global__ __launch_bounds__(64 * WM * WN, 1) void gemm_prefill2_kernel(GemmParams p) {
  constexpr int NW = WM * WN;
  static_assert(KS == 2, "stages of 64 k: an x tile's two pieces are its row halves");
  constexpr int WTN = BN / 16, XTM = BM / 16;  // 16-wide tiles per block
  constexpr int NT = WTN / WN, MT = XTM / WM;  // per wave
  constexpr int PIECES = (WTN + XTM) * KS;     // 1 KiB pieces per stage
  static_assert(PIECES % NW == 0, "pieces split evenly over the waves");
  constexpr int PPW = PIECES / NW;
  constexpr int STAGE = PIECES * 1024;
  static_assert(NT % NTB == 0 && NS >= 2 && NS <= 4, "tile groups / ring depth");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TLScope tl_scope(p.dbg_ts);
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid / WN, wn = wid % WN;
  const int KT = p.K >> 5;
  const int nk_all = KT / KS;
  const int z = blockIdx.y, nz = gridDim.y;
  const int kst0 = (nk_all * z) / nz, nk = (nk_all * (z + 1)) / nz - kst0;
  const int mblocks = (p.M + BM - 1) / BM;
  const int nwg = gridDim.x, orig = blockIdx.x, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int wgid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  const int m0 = (wgid % mblocks) * BM;
  const int nt_blk = (wgid / mblocks) * WTN;
  const char* src[PPW];
  int step[PPW];
#pragma unroll
  for (int i = 0; i < PPW; ++i) {
    const int f = wid * PPW + i;
    if (f < WTN * KS) {
      const int nt = nt_blk + f / KS, ks = f % KS;
      src[i] = reinterpret_cast<const char*>(p.wp) + (((size_t)nt * KT + KS * kst0 + ks) * 64 + lane) * 16;
      step[i] = KS * 1024;
    } else {
      const int g = f - WTN * KS;
      const int row = x_piece_row(m0 + (g >> 1) * 16, g & 1, lane, p.M);
      src[i] = reinterpret_cast<const char*>(p.x + (size_t)row * p.lda + kst0 * 64 + x_piece_col(g & 1, lane));
      step[i] = 64 * 2;
    }
  }
  const uint32_t lds0 = lds_addr_of(smem);
  const int xo[2] = {x_frag_off(0, lane), x_frag_off(1, lane)};
  auto issue_part = [&](int stage, int buf, int i0, int i1) {
    const int st = stage < nk ? stage : nk - 1;  // past the end: a clamped duplicate, never read
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
      if (i < i0 || i >= i1) continue;  // compile-time after unrolling
      const int f = wid * PPW + i;
      glds16(src[i] + (size_t)st * step[i], __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + f * 1024));
    }
  };
  auto issue = [&](int stage, int buf) { issue_part(stage, buf, 0, PPW); };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[MT];
#pragma unroll
  for (int b = 0; b < MT; ++b) ss[b] = 0.f;

#pragma unroll
  for (int s0 = 0; s0 < NS - 1; ++s0) issue(s0, s0);
  for (int t = 0; t < nk; ++t) {
    // stage t landed (this wave's pieces; the NS-2 younger stages may still be in flight), then
    // every wave's pieces (barrier) — which also retires the reads of the buffer refilled next
    if constexpr (NS == 2) asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    else if constexpr (NS == 3) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PPW) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * PPW) : "memory");
    if constexpr (SCHED < 2) issue(t + NS - 1, (t + NS - 1) % NS);
    else issue_part(t + NS - 1, (t + NS - 1) % NS, 0, PPW / 2);
    const char* sb = smem + (t % NS) * STAGE;
    // every fragment of the stage read up front (both k-steps): the second k-step's reads are in
    // flight under the first one's MFMAs instead of exposing the LDS latency per k-step
    uint4 wall[KS][NT], xall[KS][MT];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int a = 0; a < NT; ++a)
        wall[ks][a] = *reinterpret_cast<const uint4*>(sb + ((wn * NT + a) * KS + ks) * 1024 + lane * 16);
#pragma unroll
      for (int b = 0; b < MT; ++b)
        xall[ks][b] = *reinterpret_cast<const uint4*>(sb + (WTN + wm * MT + b) * 2048 + xo[ks]);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const uint4 (&wa)[NT] = wall[ks];
      const uint4 (&xb)[MT] = xall[ks];
      if constexpr (NORM == 2) {
#pragma unroll
        for (int b = 0; b < MT; ++b) {
          ss[b] = sumsq8(xb[b], ss[b]);
        }
      }
      if constexpr (SCHED == 2)
        if (ks == 1) issue_part(t + NS - 1, (t + NS - 1) % NS, PPW / 2, PPW);
      if constexpr (SCHED >= 1) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = mfma16(as_bf16x8(wa[a]), as_bf16x8(xb[b]), acc[a][b]);
      if constexpr (SCHED >= 1) __builtin_amdgcn_s_setprio(0);
    }
    // the next iteration's barrier orders these ds_reads before the buffer is refilled
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the trailing duplicate DMAs
  if (nz > 1) {
    float* part = p.slabs + (size_t)z * p.M * p.N;
    float* ssq = p.slabs + (size_t)nz * p.M * p.N + (size_t)z * p.M;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int m = m0 + wm * (BM / WM) + b * 16 + (lane & 15);
      if constexpr (NORM == 2) {
        float s2 = ss[b];
        s2 += xor16(s2);
        s2 += xor32(s2);
        if (wn == 0 && lane < 16 && m < p.M) ssq[m] = s2;
      }
      if (m < p.M) {
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          const int n = (nt_blk + wn * NT + a) * 16 + 4 * (lane >> 4);
          __builtin_nontemporal_store(acc[a][b], reinterpret_cast<f32x4*>(part + (size_t)m * p.N + n));
        }
      }
    }
    return;
  }
  float sc[MT];
#pragma unroll
  for (int b = 0; b < MT; ++b) {
    sc[b] = 1.f;
    if constexpr (NORM == 2) {
      float s2 = ss[b];
      s2 += xor16(s2);
      s2 += xor32(s2);
      sc[b] = rsqrtf(s2 / (float)p.K + p.eps);
    }
  }
  prompt_epilogue<NT, MT, EPI>(p, m0 + wm * (BM / WM), nt_blk + wn * NT, lane, [&](int a, int b) { return acc[a][b] * sc[b]; });
}

// ---- v4: 256 x 256 tile in four phases per K-tile ----
// 8 waves, wave (wr = wid >> 2, wc = wid & 3) owns n-tiles 8 wr .. 8 wr + 7 (two halves n0 / n1 of 4)
// x m-tiles 4 wc .. 4 wc + 3 (halves m0 / m1 of 2). A K-tile (BK = 64, 64 KiB: 16 W + 16 x tiles x
// 2 k-steps) is consumed in four phases, one 64 x 32 output quadrant x K = 64 (16 MFMAs) each, in
// the order (n0, m0) (n0, m1) (n1, m1) (n1, m0): phase 0 first needs W n0 + x m0, phase 1 x m1,
// phase 2 W n1, phase 3 nothing new (x m0 kept in registers). The next K-tile's LDS-DMA is issued
// in the same three groups, group g in phase g (into the other buffer, free since the previous
// K-tile's phase-0 barrier), so every piece has a whole K-tile (four phases) to land and each
// phase waits with a compile-time counted vmcnt (pieces issued after its group) + raw s_barrier —
// never vmcnt(0) in the loop (cdna_hip_programming.md §5 'The 256² 8-phase template').
// Group sizes per wave: 4 / 2 / 2 pieces -> the waits of phases 0 / 1 / 2: vmcnt(4) / (6) / (6).
// BN = 128: the same schedule on a 256 x 128 tile (wave 64 n x 64 m, 8 MFMAs per phase, 96 KiB;
// groups 3 / 2 / 1 pieces per wave -> vmcnt(3) / (4) / (5)).
template <int BN>
struct P4 {  // geometry of the 4-phase 256 x BN kernel
  static constexpr int BM = 256, KS = 2;
  static constexpr int WTN = BN / 16, XTM = BM / 16;  // W + x tiles per block (16 / 8 + 16)
  static constexpr int NWN = WTN / 2, NH = NWN / 2;   // n-tiles per wave, per n-half
  static constexpr int STAGE = (WTN + XTM) * KS * 1024;
  static constexpr int G0 = 4 * NH + 16, G1 = 16, G2 = 4 * NH;  // pieces per group (block)
  static constexpr int P0 = G0 / 8, P1 = G1 / 8, P2 = G2 / 8;  // per wave
  static constexpr int PPW = P0 + P1 + P2;
  static_assert(G0 % 8 == 0 && G2 % 8 == 0 && (BN == 256 || BN == 128), "pieces split over 8 waves");
};

// The K loop of the 4-phase kernel over K-tiles [kst0, kst0 + nk) of the block tile (m0, nt_blk),
// accumulated into acc / ss (zeroed by the caller). Ends with every DMA of this wave landed (the
// trailing clamped duplicates included); a caller that runs it again on the same LDS barriers first.
template <int BN, int NORM>
__device__ __forceinline__ void p4_kloop(const GemmParams& p, char* smem, int wid, int lane, int m0, int nt_blk,
                                         int kst0, int nk, f32x4 (&acc)[BN / 32][4], float (&ss)[4]) {
  using G = P4<BN>;
  constexpr int KS = G::KS, WTN = G::WTN, NWN = G::NWN, NH = G::NH, STAGE = G::STAGE;
  constexpr int P0 = G::P0, P1 = G::P1, P2 = G::P2, PPW = G::PPW;
  const int wr = wid >> 2, wc = wid & 3;
  const int KT = p.K >> 5;
  // this wave's pieces: entries of the group lists (block-local tile, k-step; W or x)
  //   group 0: the n0 W tiles of both wave rows, then x tiles {4c, 4c + 1}, x 2 k-steps
  //   group 1: x tiles {4c + 2, 4c + 3} x 2
  //   group 2: the n1 W tiles x 2
  const char* src[PPW];
  int step[PPW];
  uint32_t dst[PPW];
  const uint32_t lds0 = lds_addr_of(smem);
  const int xo[2] = {x_frag_off(0, lane), x_frag_off(1, lane)};
#pragma unroll
  for (int i = 0; i < PPW; ++i) {
    int e, isw, t;
    if (i < P0) {
      e = wid * P0 + i;
      if (e < 4 * NH) {
        isw = 1;
        const int tw = e >> 1;
        t = (tw / NH) * NWN + tw % NH;
      } else {
        isw = 0;
        const int tile8 = (e - 4 * NH) >> 1;
        t = 4 * (tile8 >> 1) + (tile8 & 1);
      }
    } else if (i < P0 + P1) {
      e = wid * P1 + (i - P0);
      isw = 0;
      const int tile8 = e >> 1;
      t = 4 * (tile8 >> 1) + 2 + (tile8 & 1);
    } else {
      e = wid * P2 + (i - P0 - P1);
      isw = 1;
      const int tw = e >> 1;
      t = (tw / NH) * NWN + NH + tw % NH;
    }
    const int ks = e & 1;
    if (isw) {
      src[i] = reinterpret_cast<const char*>(p.wp) + (((size_t)(nt_blk + t) * KT + 2 * kst0 + ks) * 64 + lane) * 16;
      step[i] = KS * 1024;
      dst[i] = (uint32_t)((t * KS + ks) * 1024);
    } else {
      const int row = x_piece_row(m0 + t * 16, ks, lane, p.M);  // (an x tile's two pieces are its row halves, see x_piece_row)
      src[i] = reinterpret_cast<const char*>(p.x + (size_t)row * p.lda + kst0 * 64 + x_piece_col(ks, lane));
      step[i] = 64 * 2;
      dst[i] = (uint32_t)((WTN * KS + t * KS + ks) * 1024);
    }
  }
  auto issue_group = [&](int g, int stage, int buf) {
    const int st = stage < nk ? stage : nk - 1;  // past the end: clamped duplicates, never read
    const int i0 = g == 0 ? 0 : g == 1 ? P0 : P0 + P1, i1 = g == 0 ? P0 : g == 1 ? P0 + P1 : PPW;
#pragma unroll
    for (int i = 0; i < PPW; ++i) {
      if (i < i0 || i >= i1) continue;
      glds16(src[i] + (size_t)st * step[i], __builtin_amdgcn_readfirstlane(lds0 + buf * STAGE + dst[i]));
    }
  };
  uint4 wf[KS][NH], x0[KS][2], x1[KS][2];
  auto read_w = [&](const char* sb, int half) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int a = 0; a < NH; ++a)
        wf[ks][a] = *reinterpret_cast<const uint4*>(sb + ((wr * NWN + half * NH + a) * KS + ks) * 1024 + lane * 16);
  };
  auto read_x = [&](const char* sb, int half, uint4 (&xf)[KS][2]) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        xf[ks][b] = *reinterpret_cast<const uint4*>(sb + (WTN + wc * 4 + half * 2 + b) * 2048 + xo[ks]);
    // folded RMSNorm: x^2 of the rows in packed bf16 dot products (v_dot2_f32_bf16: one op per 2
    // elements, no unpack), and only in wave row 0 — wave row 1 reads the same x tiles; the row
    // sums reach it through LDS in p4_finish. (The unpack + FMA form in both wave rows cost the
    // folded-norm GEMMs ~20 % against the same tile without the norm: Llama-3-8B gate_up at
    // 2048 rows 472 vs 399 us.)
    if constexpr (NORM == 2) {
      if (wr == 0) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int b = 0; b < 2; ++b) ss[half * 2 + b] = sumsq8(xf[ks][b], ss[half * 2 + b]);
      }
    }
  };
  auto quadrant = [&](int nh, int mh, const uint4 (&xf)[KS][2]) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int a = 0; a < NH; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[nh * NH + a][mh * 2 + b] = mfma16(as_bf16x8(wf[ks][a]), as_bf16x8(xf[ks][b]), acc[nh * NH + a][mh * 2 + b]);
    __builtin_amdgcn_s_setprio(0);
  };
  issue_group(0, 0, 0);
  issue_group(1, 0, 0);
  issue_group(2, 0, 0);
  for (int t = 0; t < nk; ++t) {
    const int buf = t & 1;
    const char* sb = smem + buf * STAGE;
    // phase 0: (n0, m0) — group 0 of this K-tile (groups 1, 2 issued after it)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(P1 + P2) : "memory");
    read_w(sb, 0);
    read_x(sb, 0, x0);
    issue_group(0, t + 1, buf ^ 1);
    quadrant(0, 0, x0);
    // phase 1: (n0, m1) — group 1 (issued after it: group 2 of this tile, group 0 of the next)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(P2 + P0) : "memory");
    read_x(sb, 1, x1);
    issue_group(1, t + 1, buf ^ 1);
    quadrant(0, 1, x1);
    // phase 2: (n1, m1) — group 2 (issued after it: groups 0, 1 of the next tile)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(P0 + P1) : "memory");
    read_w(sb, 1);
    issue_group(2, t + 1, buf ^ 1);
    quadrant(1, 1, x1);
    // phase 3: (n1, m0) from registers
    quadrant(1, 0, x0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the trailing duplicate DMAs
}

// the epilogue of a finished 256 x BN block tile straight from the accumulators (deferred row scale)
// (NORM == 2: the row sums of squares are in wave row 0's ss; wave row 1 gets them through the 1 KiB
// LDS area P4_ROWSS past the ring — block-uniform call, one barrier)
constexpr int P4_ROWSS = 16;  // byte offset past the 2-stage ring
template <int BN, int EPI, int NORM, int NTB>
__device__ __forceinline__ void p4_finish(const GemmParams& p, char* smem, int wid, int lane, int m0, int nt_blk,
                                          f32x4 (&acc)[BN / 32][4], const float (&ss)[4]) {
  constexpr int NWN = P4<BN>::NWN;
  const int wr = wid >> 2, wc = wid & 3;
  float rs[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (NORM == 2) {
    float* rows = reinterpret_cast<float*>(smem + 2 * P4<BN>::STAGE + P4_ROWSS);
    if (wr == 0) {
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        float s2 = ss[b];
        s2 += xor16(s2);
        s2 += xor32(s2);
        rs[b] = s2;
        if (lane < 16) rows[wc * 64 + b * 16 + lane] = s2;
      }
    }
    lds_barrier();
    if (wr != 0) {
#pragma unroll
      for (int b = 0; b < 4; ++b) rs[b] = rows[wc * 64 + b * 16 + (lane & 15)];
    }
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) rs[b] = NORM == 2 ? rsqrtf(rs[b] / (float)p.K + p.eps) : 1.f;
  prompt_epilogue<NWN, 4, EPI>(p, m0 + wc * 64, nt_blk + wr * NWN, lane, [&](int a, int b) { return acc[a][b] * rs[b]; });
}

template <int BN, int EPI, int NORM, int NTB>
__global__ __launch_bounds__(512, 1) void gemm_prefill4_kernel(GemmParams p) {
  using G = P4<BN>;
  constexpr int BM = G::BM, WTN = G::WTN, NWN = G::NWN;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TLScope tl_scope(p.dbg_ts);
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wid >> 2, wc = wid & 3;
  const int nk_all = p.K >> 6;
  const int z = blockIdx.y, nz = gridDim.y;
  const int kst0 = (nk_all * z) / nz, nk = (nk_all * (z + 1)) / nz - kst0;
  const int mblocks = (p.M + BM - 1) / BM;
  const int nwg = gridDim.x, orig = blockIdx.x, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int wgid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  const int m0 = (wgid % mblocks) * BM;
  const int nt_blk = (wgid / mblocks) * WTN;
  f32x4 acc[NWN][4];
#pragma unroll
  for (int a = 0; a < NWN; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[4] = {0.f, 0.f, 0.f, 0.f};
  p4_kloop<BN, NORM>(p, smem, wid, lane, m0, nt_blk, kst0, nk, acc, ss);
  if (nz > 1) {
    float* part = p.slabs + (size_t)z * p.M * p.N;
    float* ssq = p.slabs + (size_t)nz * p.M * p.N + (size_t)z * p.M;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int m = m0 + wc * 64 + b * 16 + (lane & 15);
      if constexpr (NORM == 2) {
        float s2 = ss[b];
        s2 += xor16(s2);
        s2 += xor32(s2);
        if (wr == 0 && lane < 16 && m < p.M) ssq[m] = s2;
      }
      if (m < p.M) {
#pragma unroll
        for (int a = 0; a < NWN; ++a) {
          const int n = (nt_blk + wr * NWN + a) * 16 + 4 * (lane >> 4);
          __builtin_nontemporal_store(acc[a][b], reinterpret_cast<f32x4*>(part + (size_t)m * p.N + n));
        }
      }
    }
    return;
  }
  p4_finish<BN, EPI, NORM, NTB>(p, smem, wid, lane, m0, nt_blk, acc, ss);
}

// ---- persistent form of the 4-phase kernel: whole rounds + a K-split last round, one launch ----
// A tile grid of T tiles on G CUs takes ceil(T / G) rounds and the last one runs R = T mod G tiles
// on a fraction of the chip (Llama-3-8B gate_up at 2048 rows: 896 tiles = 3 rounds + 128 tiles; o /
// down: 128 tiles = half the chip). Here G = #CU resident blocks (one per CU: the LDS ring) run the
// T - R tiles of the whole rounds in order — block g takes tile r * G + g in round r, so each XCD
// keeps working on 4 weight panels x all m-blocks at the same K position, as the tile grid does
// (the L2 reuse a free (tile, K-tile) stream-K split loses: its blocks sit at unrelated K offsets
// and it measured 1.3x SLOWER than the tile grid, profiles/r6_prefill_stream_k.log) — and then
// the R tail tiles as S K slices each: unit u = (S - 1 - c) * R + j is slice c of tail tile j, block
// g takes units g, g + G, ... (the launcher's S keeps R S <= G, one round: Llama-3-8B gate_up / down /
// o_proj at 2048 rows, S = 2; a forced larger S runs several rounds), so the blocks of one XCD
// again share panels and K positions.
// Slices c > 0 publish their fp32 partial (+ the x sums of squares of the folded RMSNorm) to the
// unit's slot with device-coherent stores and count in on the tile's ticket; slice 0 (the owner)
// waits for the S - 1 tickets, adds the partials in slice order (bit-reproducible), runs the epilogue
// and clears the ticket. Every block takes its units in order and all of the later slices come
// before the owners, so a slice never waits: an owner's partials are either done or being computed
// by a resident block that needs nothing from anyone; the poll is bounded all the same (give-up:
// bit 64 of the fault word, garbage, never a hang).
constexpr int P4SK_SPIN = 1 << 20;

template <int BN>
__host__ __device__ constexpr int p4sk_slot_floats() {
  return (P4<BN>::NWN * 4 + 1) * 512 * 4;  // 512 threads x (NWN x 4 accumulators + the row sums) f32x4
}

// slot traffic: lane part in ONE VGPR (tid * 16), the accumulator index in the scalar offset (a
// per-index VGPR offset is loop-invariant, gets hoisted over the K loop and spills the 256-wide tile)
__device__ __forceinline__ void p4sk_st(float* slot, int tid, int j, f32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, rsrc_of(slot), (uint32_t)tid * 16, j * 8192, 16 /* sc1 */);
}
__device__ __forceinline__ f32x4 p4sk_ld(const float* slot, int tid, int j) {
  return __builtin_amdgcn_raw_buffer_load_b128(rsrc_of(slot), (uint32_t)tid * 16, j * 8192, 16 /* sc1 */);
}

template <int BN, int EPI, int NORM, int NTB>
__global__ __launch_bounds__(512, 1) void gemm_prefill4sk_kernel(GemmParams p0, int tiles, int S) {
  using G = P4<BN>;
  constexpr int BM = G::BM, WTN = G::WTN, NWN = G::NWN, NACC = NWN * 4;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TLScope tl_scope(p0.dbg_ts);
  const int KT = p0.K >> 6;
  const int mblocks = (p0.M + BM - 1) / BM;
  const int nwg = gridDim.x, orig = blockIdx.x, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  // XCD-aware: consecutive g (tiles of one weight column panel, m-blocks fastest) on one XCD
  const int g = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  const int full = tiles / nwg, R = tiles - full * nwg;
  const int RS = R * S, nseg = full + (g < RS ? (RS - g + nwg - 1) / nwg : 0);
  const auto kp0 = (const GemmParams __attribute__((address_space(4)))*)(__builtin_amdgcn_kernarg_segment_ptr());
  for (int i = 0; i < nseg; ++i) {  // block-uniform
    if (i > 0) __builtin_amdgcn_s_barrier();  // the previous tile's LDS reads + DMAs are done
    // the parameters re-read from the kernel-argument segment per tile: hoisted out of this loop,
    // the epilogue's pointers would sit in SGPRs across the K loop (SGPR spills into VGPR lanes);
    // thread ids laundered likewise (no lane-derived epilogue / slot address stays live across it)
    auto kp = kp0;
    asm volatile("" : "+s"(kp));
    const GemmParams& p = *(const GemmParams*)kp;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    int tile = i * nwg + g, k0 = 0, k1 = KT, c = -1, j = 0, u = 0;
    if (i >= full) {  // tail unit u: slice c of tail tile j, the later slices first (the owners last)
      u = g + (i - full) * nwg;
      j = u % R;
      c = S - 1 - u / R;
      tile = full * nwg + j;
      k0 = (KT * c) / S;
      k1 = (KT * (c + 1)) / S;
    }
    const int m0 = (tile % mblocks) * BM, nt_blk = (tile / mblocks) * WTN;
    f32x4 acc[NWN][4];
#pragma unroll
    for (int a = 0; a < NWN; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float ss[4] = {0.f, 0.f, 0.f, 0.f};
    if (c > 0) {  // a later K slice of a tail tile: publish, count in (its own copy of the K loop: with
                  // one copy shared by this path and the owner's the allocator spills the accumulators)
      p4_kloop<BN, NORM>(p, smem, wid, lane, m0, nt_blk, k0, k1 - k0, acc, ss);
      float* slot = p.slabs + (size_t)u * p4sk_slot_floats<BN>();  // u < R (S - 1): one slot per unit
#pragma unroll
      for (int e = 0; e < NACC; ++e) p4sk_st(slot, tid, e, acc[e >> 2][e & 3]);
      if constexpr (NORM == 2) p4sk_st(slot, tid, NACC, f32x4{ss[0], ss[1], ss[2], ss[3]});
      drain_stores();
      __syncthreads();
      if (tid == 0) __hip_atomic_fetch_add(p.counters + j, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      continue;
    }
    p4_kloop<BN, NORM>(p, smem, wid, lane, m0, nt_blk, k0, k1 - k0, acc, ss);
    if (c == 0 && S > 1) {  // the owner of a split tail tile: wait for slices 1 .. S - 1, add in order
      if (tid == 0) {
        int spins = 0;
        while (__hip_atomic_load(p.counters + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (uint32_t)(S - 1)) {
          if (++spins > P4SK_SPIN) {
            if (p.fault != nullptr) atomicOr(p.fault, 64u);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
      __syncthreads();
      for (int cc = 1; cc < S; ++cc) {
        const float* slot = p.slabs + (size_t)((S - 1 - cc) * R + j) * p4sk_slot_floats<BN>();
        // a quarter of the accumulators per round trip (the loads' registers: 32 / 16 per lane)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          f32x4 v[NACC / 4];
#pragma unroll
          for (int e = 0; e < NACC / 4; ++e) v[e] = p4sk_ld(slot, tid, h * NACC / 4 + e);
#pragma unroll
          for (int e = 0; e < NACC / 4; ++e) acc[(h * NACC / 4 + e) >> 2][(h * NACC / 4 + e) & 3] += v[e];
          asm volatile("" ::: "memory");
        }
        if constexpr (NORM == 2) {
          const f32x4 s4 = p4sk_ld(slot, tid, NACC);
          ss[0] += s4[0]; ss[1] += s4[1]; ss[2] += s4[2]; ss[3] += s4[3];
        }
      }
      if (tid == 0) __hip_atomic_store(p.counters + j, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    p4_finish<BN, EPI, NORM, NTB>(p, smem, wid, lane, m0, nt_blk, acc, ss);
  }
}

// Split-K combine: one wave per (16 rows, NTB tiles): the slices' partials summed in slice
// order, the row scale from the summed slice sums of squares, then the shared epilogue. The
// slices' loads go out in groups of ZG (clamped index, masked add) so a combine costs one memory
// round trip per ZG slices instead of one per slice.
template <int EPI, int NORM, int NTB>
__global__ __launch_bounds__(256) void prefill_reduce_kernel(GemmParams p, int nz) {
  constexpr int ZG = 8;
  TLScope tl_scope(p.dbg_ts);
  const int lane = threadIdx.x & 63;
  const int grp = blockIdx.x * 4 + (threadIdx.x >> 6);  // (row block, tile group), tile group fastest
  const int ngrp = p.N / (16 * NTB);
  if (grp >= ((p.M + 15) / 16) * ngrp) return;  // wave-uniform
  const int m = (grp / ngrp) * 16 + (lane & 15);
  const int nt0 = (grp % ngrp) * NTB;
  const int nsub = 4 * (lane >> 4);
  const int mm = m < p.M ? m : p.M - 1;
  f32x4 v[NTB];
#pragma unroll
  for (int j = 0; j < NTB; ++j) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float s2 = 0.f;
  for (int z0 = 0; z0 < nz; z0 += ZG) {
    f32x4 r[ZG][NTB];
    float q[ZG];
#pragma unroll
    for (int u = 0; u < ZG; ++u) {
      const int z = min(z0 + u, nz - 1);
      const float* part = p.slabs + (size_t)z * p.M * p.N + (size_t)mm * p.N;
#pragma unroll
      for (int j = 0; j < NTB; ++j) r[u][j] = *reinterpret_cast<const f32x4*>(part + (nt0 + j) * 16 + nsub);
      q[u] = NORM == 2 ? p.slabs[(size_t)nz * p.M * p.N + (size_t)z * p.M + mm] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < ZG; ++u) {
      if (z0 + u < nz) {
#pragma unroll
        for (int j = 0; j < NTB; ++j) v[j] += r[u][j];
        if constexpr (NORM == 2) s2 += q[u];
      }
    }
  }
  if constexpr (NORM == 2) {
    const float sc = rsqrtf(s2 / (float)p.K + p.eps);
#pragma unroll
    for (int j = 0; j < NTB; ++j) v[j] *= sc;
  }
  epilogue<NTB, EPI, false>(p, v, m, nt0, nsub, EpiPre<NTB>{}, m < p.M);
}

// the combine launch for p.splitk-free callers (gemm_mid.hip)
template <int EPI, int NORM, int NTB>
void launch_prefill_reduce(const GemmParams& p, int nz, hipStream_t st) {
  const int groups = ((p.M + 15) / 16) * (p.N / (16 * NTB));
  GemmParams r = p;
  r.dbg_ts = tl_take("prefill_reduce", (groups + 3) / 4);
  hipLaunchKernelGGL((prefill_reduce_kernel<EPI, NORM, NTB>), dim3((groups + 3) / 4), dim3(256), 0, st, r, nz);
}
#define VG_RED_INST(E)                                                                  \
  template void launch_prefill_reduce<E, 0, 1>(const GemmParams&, int, hipStream_t);   \
  template void launch_prefill_reduce<E, 2, 1>(const GemmParams&, int, hipStream_t);
VG_RED_INST(EPI_BF16)
VG_RED_INST(EPI_F32)
VG_RED_INST(EPI_SILU)
VG_RED_INST(EPI_QKV)
template void launch_prefill_reduce<EPI_GLU, 0, 1>(const GemmParams&, int, hipStream_t);
#undef VG_RED_INST

template <int EPI, int NORM, int NTB, int BM = 256, int BN = 128, int WM = 4, int WN = 2, int NS = 3, int SCHED = 0,
          int KS = 2>
static void launch_prefill2_one(const GemmParams& p, int nz, hipStream_t st) {
  constexpr int STAGE = (BN / 16 + BM / 16) * KS * 1024;
  const int blocks = ((p.M + BM - 1) / BM) * (p.N / BN);
  GemmParams q = p;
  if (q.dbg_ts == nullptr) q.dbg_ts = tl_take("gemm_prefill2", blocks * nz);
  auto kern = gemm_prefill2_kernel<BM, BN, WM, WN, NS, EPI, NORM, NTB, SCHED, KS>;
  static bool attr = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               NS * STAGE) == hipSuccess;
  }();
  (void)attr;
  hipLaunchKernelGGL(kern, dim3(blocks, nz), dim3(64 * WM * WN), NS * STAGE, st, q);
  if (nz > 1) {
    const int groups = ((p.M + 15) / 16) * (p.N / (16 * NTB));
    GemmParams r = p;
    r.dbg_ts = tl_take("prefill_reduce", (groups + 3) / 4);
    hipLaunchKernelGGL((prefill_reduce_kernel<EPI, NORM, NTB>), dim3((groups + 3) / 4), dim3(256), 0, st, r, nz);
  }
}

template <int EPI, int NORM, int NTB, int BM = 256, int BN = 128, int WM = 4, int WN = 2, int NS = 3, int KS = 2>
static void launch_prefill2_cfg(const GemmParams& p, int nz, hipStream_t st) {
  // MFMAs at raised priority (schedule 1): +5-7 % on the 256 x 256 tile, neutral on 256 x 128; the
  // split DMA issue was neutral to negative (profiles/r2_prefill_gemm_sched.log)
  launch_prefill2_one<EPI, NORM, NTB, BM, BN, WM, WN, NS, 1, KS>(p, nz, st);
}

template <int EPI, int NORM, int NTB, int BN = 256>
static void launch_prefill4_cfg(const GemmParams& p, int nz, hipStream_t st) {
  constexpr int STAGE = (BN / 16 + 16) * 2 * 1024;
  const int blocks = ((p.M + 255) / 256) * (p.N / BN);
  GemmParams q = p;
  if (q.dbg_ts == nullptr) q.dbg_ts = tl_take("gemm_prefill4", blocks * nz);
  auto kern = gemm_prefill4_kernel<BN, EPI, NORM, NTB>;
  constexpr int LDS = 2 * STAGE + P4_ROWSS + 1024;  // ring + the folded norm's row sums
  static bool attr = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               LDS) == hipSuccess;
  }();
  (void)attr;
  hipLaunchKernelGGL(kern, dim3(blocks, nz), dim3(512), LDS, st, q);
  if (nz > 1) {
    const int groups = ((p.M + 15) / 16) * (p.N / (16 * NTB));
    GemmParams r = p;
    r.dbg_ts = tl_take("prefill_reduce", (groups + 3) / 4);
    hipLaunchKernelGGL((prefill_reduce_kernel<EPI, NORM, NTB>), dim3((groups + 3) / 4), dim3(256), 0, st, r, nz);
  }
}

static int cu_count() {
  static const int n = [] {
    int dev = 0, c = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      c = 0;
    return c;
  }();
  return n;
}

// persistent 4-phase kernel (whole rounds + the K-split tail), one block per CU; slices = the tail's K
// slices (0: G / R, at least 4 K-tiles each, at most 8). false = not taken (no tail to split, no
// tickets / slot room)
template <int EPI, int NORM, int NTB, int BN>
static bool launch_prefill4sk_cfg(const GemmParams& p, int slices, int max_counters, size_t slab_bytes,
                                  hipStream_t st) {
  constexpr int STAGE = (BN / 16 + 16) * 2 * 1024;
  const int tiles = ((p.M + 255) / 256) * (p.N / BN);
  const int G = cu_count();
  if (G <= 0 || p.counters == nullptr || p.slabs == nullptr) return false;
  const int R = tiles % G, KT = p.K / 64;
  if (R == 0) return false;  // whole rounds: the tile grid is the same schedule
  // S (0: the launcher's choice): the tail in ONE round, S = G / R slices (<= 8). More slices than fit
  // one round (forced, or a tuner candidate) run in several: measured slower at every shape tried but
  // Llama-3-8B qkv_proj (192 tiles x 8 slices: 115 vs 123 us, where the split-K 6 grid + reduce is 108),
  // every contributor pays the drain of its 270 KB partial (r6_prefill_persistent_tail.log)
  int S = slices > 0 ? slices : (G / R > 8 ? 8 : G / R);
  while (S > 1 && KT / S < 4) --S;
  if (S < 1 || R > max_counters || (size_t)R * (S - 1) * p4sk_slot_floats<BN>() * 4 > slab_bytes) return false;
  GemmParams q = p;
  if (q.dbg_ts == nullptr) q.dbg_ts = tl_take("gemm_prefill4sk", G);
  auto kern = gemm_prefill4sk_kernel<BN, EPI, NORM, NTB>;
  constexpr int LDS = 2 * STAGE + P4_ROWSS + 1024;  // ring + the folded norm's row sums
  static bool attr = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                               LDS) == hipSuccess;
  }();
  (void)attr;
  hipLaunchKernelGGL(kern, dim3(G), dim3(512), LDS, st, q, tiles, S);
  return true;
}

template <int BM, int BN, int EPI, int NORM, int NTB>
static void launch_prefill_cfg(const GemmParams& p, int nz, hipStream_t st) {
  constexpr int STAGE = (BN / 16 + BM / 16) * 2 * 1024;
  const int blocks = ((p.M + BM - 1) / BM) * (p.N / BN);
  GemmParams q = p;
  if (q.dbg_ts == nullptr) q.dbg_ts = tl_take("gemm_prefill", blocks * nz);
  hipLaunchKernelGGL((gemm_prefill_kernel<BM, BN, EPI, NORM, NTB>), dim3(blocks, nz), dim3(256), 2 * STAGE, st, q);
  if (nz > 1) {
    const int groups = ((p.M + 15) / 16) * (p.N / (16 * NTB));
    GemmParams r = p;
    r.dbg_ts = tl_take("prefill_reduce", (groups + 3) / 4);
    hipLaunchKernelGGL((prefill_reduce_kernel<EPI, NORM, NTB>), dim3((groups + 3) / 4), dim3(256), 0, st, r, nz);
  }
}

// Split-K partials leave with non-temporal stores: dirty fp32 slabs in L2 are written back at the
// kernel boundary and held the next launch back 2-4 us (prefill-step timeline, r4).
//
// The launcher's own choice of tile and K slices: the cheapest form by a fitted cost (us),
//     e + a x rounds + b x K-tiles of the busiest CU + w x MB of weights + o x MB of output
//     [+ c + d x MB of partials: a K-split grid and its combine launch]
// with rounds = blocks over what the CUs hold, rounded up. A large tile has the highest rate and the worst last round, the small ones
// the shortest chain; splitting K fills the chip for few tiles and costs a pass over the partials. Fitted (non-negative least squares
// on relative errors) to 26 shapes (N 512 .. 28672, K 512 .. 14336) x 15 row counts 65 .. 2048 on cold weights, apart with the row
// scale of a folded norm; rms error 3 to 6 % per form (the persistent ones 11). The choice takes 1.008 of the time of the best form there
// (geometric mean) and 0.92 of hipBLASLt's; without 64 x 64 1.054, without 128 x 64 1.021, without 128 x 128 1.016, without any other one of
// them 1.009 to 1.011. us before the four-wave forms (gemm_prompt.h) -> now: 1536 x 1536 at 256 rows 16.6 -> 12.5, 2048 x 1536 at 448
// 17.1 -> 12.6, 17920 x 1536 at 448 46.8 -> 38.8, 4352 x 1024 at 2048 36.6 -> 30.3, 1024 x 4096 at 1024 32.2 -> 24.0.
// cut > 0: that many K slices and none of the persistent forms
static PrefillForm choose_prefill_form(int M, int N, int K, bool norm, bool rows16, bool slabs, size_t slab_bytes, bool counters, int cut = 0) {
  struct Cost {
    float e, a, b, c, d, w, o;
  };
  struct Tile {
    int code, bm, bn, per_cu;
    Cost cost[2];  // plain, with a folded norm
  };
  static constexpr Tile tiles[] = {
      {5220, 64, 64, 2, {{6.58f, 0.615f, 0.232f, 2.7f, 0.566f, 0.034f, 0.063f}, {6.96f, 0.657f, 0.238f, 2.73f, 0.514f, 0.035f, 0.105f}}},
      {5340, 96, 128, 1, {{6.19f, 2.54f, 0.473f, 2.84f, 0.432f, 0.031f, 0.187f}, {7.24f, 2.94f, 0.49f, 1.8f, 0.422f, 0.024f, 0.224f}}},
      {5380, 96, 256, 1, {{9.21f, 2.5f, 0.737f, 0.f, 0.f, 0.034f, 0.f}, {11.5f, 2.48f, 0.757f, 0.f, 0.f, 0.02f, 0.f}}},
      {5580, 160, 256, 1, {{9.64f, 6.38f, 0.948f, 0.f, 0.f, 0.018f, 0.f}, {15.4f, 5.08f, 0.986f, 0.f, 0.f, 0.005f, 0.f}}},
      {5640, 192, 128, 1, {{8.36f, 3.99f, 0.624f, 0.f, 0.f, 0.012f, 0.139f}, {9.96f, 5.92f, 0.67f, 0.f, 0.f, 0.f, 0.f}}},
      {5680, 192, 256, 1, {{14.5f, 1.91f, 1.25f, 0.f, 0.f, 0.007f, 0.f}, {19.4f, 1.41f, 1.25f, 0.f, 0.f, 0.f, 0.f}}},
      {641, 128, 64, 1, {{5.18f, 1.15f, 0.374f, 3.25f, 0.492f, 0.003f, 0.402f}, {5.11f, 1.5f, 0.408f, 3.32f, 0.454f, 0.017f, 0.445f}}},
      {1281, 128, 128, 1, {{5.48f, 2.17f, 0.52f, 3.05f, 0.42f, 0.012f, 0.362f}, {5.8f, 2.3f, 0.641f, 2.74f, 0.414f, 0.01f, 0.367f}}},
      {768, 256, 128, 1, {{7.23f, 1.58f, 0.811f, 1.76f, 0.461f, 0.f, 0.408f}, {7.75f, 2.09f, 0.916f, 1.16f, 0.444f, 0.f, 0.414f}}},
      {1024, 256, 256, 1, {{8.56f, 4.43f, 1.26f, 0.f, 0.458f, 0.f, 0.39f}, {8.52f, 4.65f, 1.39f, 0.f, 0.445f, 0.f, 0.427f}}}};
  // the persistent four-phase forms: e + b x K-tiles in whole rounds, then r x K-tiles of the rest [+ c + d x (slices - 1): their meeting]
  struct Persistent {
    int code, bn;
    struct {
      float e, b, r, c, d, w, o;
    } cost[2];
  };
  static constexpr Persistent persistent[] = {
      {1025, 256, {{0.f, 0.638f, 1.15f, 18.8f, 4.42f, 0.231f, 0.819f}, {0.f, 0.75f, 1.27f, 19.9f, 4.63f, 0.217f, 0.824f}}},
      {769, 128, {{6.94f, 0.703f, 0.815f, 7.04f, 2.78f, 0.051f, 0.538f}, {7.24f, 0.71f, 0.841f, 7.87f, 2.85f, 0.11f, 0.631f}}}};
  static constexpr int slices[] = {1, 2, 3, 4, 6, 8};
  const int cus = cu_count() > 0 ? cu_count() : 256, nk = K / 64;
  const float wmb = 2e-6f * (float)N * (float)K, omb = 2e-6f * (float)M * (float)N;
  auto over = [](int64_t x, int64_t y) { return (int)((x + y - 1) / y); };
  PrefillForm best{641, 1, 1e30f};
  auto take = [&](int code, int nz, float t) {
    if (t < best.us) best = PrefillForm{code, nz, t};
  };
  for (const Tile& t : tiles) {
    if (N % t.bn != 0 || (t.code >= 5000 && !rows16)) continue;
    const Cost& x = t.cost[norm ? 1 : 0];
    const bool sliced = x.d > 0.f && !(t.bm == 256 && M >= 512);  // (the four-phase tiles of long steps are split by the persistent forms)
    auto consider = [&](int nz) {
      const int64_t blocks = (int64_t)over(M, t.bm) * (N / t.bn) * nz;
      if (nz > 1 && (nk / nz < 4 || !slabs || ((size_t)nz * M * N + (size_t)nz * M) * 4 > slab_bytes)) return;
      take(t.code, nz, x.e + x.a * over(blocks, (int64_t)cus * t.per_cu) + x.b * over(blocks, cus) * over(nk, nz) + x.w * wmb + x.o * omb +
                           (nz > 1 ? x.c + x.d * 2.f * nz * omb : 0.f));
    };
    if (cut > 0) {
      if (cut == 1 || x.d > 0.f) consider(cut);
      continue;
    }
    for (int nz : slices)
      if (nz == 1 || (sliced && (int64_t)over(M, t.bm) * (N / t.bn) * nz <= 600)) consider(nz);
  }
  if (M >= 512 && slabs && counters && cut == 0) {
    for (const Persistent& t : persistent) {
      const auto& x = t.cost[norm ? 1 : 0];
      const int n = N % t.bn == 0 ? over(M, 256) * (N / t.bn) : 0, rest = n % cus;
      if (rest == 0) continue;
      int S = cus / rest > 8 ? 8 : cus / rest;
      while (S > 1 && nk / S < 4) --S;
      take(t.code, 0, x.e + x.b * (n / cus) * nk + x.r * nk / S + (S > 1 ? x.c + x.d * (S - 1) : 0.f) + x.w * wmb + x.o * omb);
    }
  }
  return best;
}

// Products with int4 weights: how each sum over K is cut. An output is the sum of `nz` chains over equal stretches of 64-k tiles, whichever
// tile computes it, on a bf16 copy (here) or on the int4 weights themselves (gemm_prompt_q4.hip), so the cut alone decides the last bits of
// the result. It has costs of its own, which stay as they are when those above are fitted anew: with random int4 weights, whose values have
// a mean, nearly all of a token's last hidden state lies along one direction, and on which side of zero it comes to lie there can rest on
// the rounding of a sum (a cut chosen by the costs above: in 8 of 400 steps some token's cached keys and values had the opposite sign).
// code 641 .. 1281: chains of a tile; 769 / 1025: of the persistent forms' slices, or (nz 0: more tiles than CUs) the persistent form
// itself; 0: the tile kernels of gemm_decode.h, one chain; -1: the K-split kernels there. tiles_only: not those because the rows are few.
PrefillForm q4_cut(int M, int N, int K, bool norm, bool rows16, bool tiles_only, size_t slab_bytes) {
  struct Tile {
    int code, bm, bn;
    float a, b, c, d;  // rounds x (a + b x K-tiles) [+ c + d x MB of partials]
  };
  struct Costs {
    Tile tiles[4];
    float n64[2], n128[2];   // whole, per K-tile and block of a CU
    float p256[4], p128[4];  // persistent: the last round whole, per K-tile, and of its K slices
  };
  static constexpr Costs sets[2] = {{{{1024, 256, 256, 10.2f, 1.33f, 1.5f, 0.49f},
                                      {768, 256, 128, 7.1f, 1.00f, 1.6f, 0.56f},
                                      {1281, 128, 128, 5.8f, 0.61f, 2.8f, 0.57f},
                                      {641, 128, 64, 5.0f, 0.50f, 2.9f, 0.62f}},
                                     {5.0f, 0.54f}, {6.0f, 0.77f}, {13.4f, 1.61f, 13.6f, 2.4f}, {10.6f, 1.07f, 5.6f, 1.5f}},
                                    {{{1024, 256, 256, 16.2f, 1.52f, -3.1f, 0.485f},
                                      {768, 256, 128, 11.7f, 1.13f, -0.8f, 0.506f},
                                      {1281, 128, 128, 9.0f, 0.705f, 2.4f, 0.395f},
                                      {641, 128, 64, 7.6f, 0.585f, 3.0f, 0.412f}},
                                     {10.5f, 0.548f}, {12.0f, 0.78f}, {22.0f, 1.59f, 13.7f, 4.2f}, {15.3f, 1.175f, 6.3f, 2.4f}}};
  const bool longer = M >= 128 || tiles_only || (rows16 && (K >= 2560 || (int64_t)N * K >= 8 * 1024 * 1024));
  if (!longer || N % 64 != 0 || K % 64 != 0) return PrefillForm{-1, 0, 0.f};
  const Costs& cs = sets[norm ? 1 : 0];
  static constexpr int slices[] = {1, 2, 3, 4, 6, 8};
  const int cus = cu_count() > 0 ? cu_count() : 256, nk = K / 64;
  auto over = [](int64_t x, int y) { return (int)((x + y - 1) / y); };
  PrefillForm best{641, 1, 1e30f};
  auto take = [&](int code, int nz, float t) {
    if (t < best.us) best = PrefillForm{code, nz, t};
  };
  if (K % 256 == 0 && N / 16 < 1024) {  // 64 x 64 tiles, weights in registers
    const int rounds = over((int64_t)over(M, 64) * (N / 64), cus);
    const bool tiles = M >= 128 || (int64_t)(N / 64) * over(M, 64) >= 128;
    take(tiles ? 0 : -1, 1, norm && K >= 768 ? 5.2f + rounds * (3.58f + 0.591f * nk) : rounds * (4.6f + 0.354f * nk));
  }
  for (const Tile& t : cs.tiles) {
    if (N % t.bn != 0) continue;
    for (int nz : slices) {
      const int64_t blocks = (int64_t)over(M, t.bm) * (N / t.bn) * nz;
      const int rounds = over(blocks, cus);
      if (nz > 1 && (rounds > 1 || nk / nz < 4 || ((size_t)nz * M * N + (size_t)nz * M) * 4 > slab_bytes)) continue;
      const float mb = (float)nz * M * N * 4e-6f;
      take(t.code, nz, rounds * (t.a + t.b * over(nk, nz)) + (nz > 1 ? t.c + t.d * mb : 0.f));
    }
  }
  const int n64 = over((int64_t)over(M, 128) * (N / 64), cus), n128 = N % 128 == 0 ? over((int64_t)over(M, 128) * (N / 128), cus) : 0;
  if (n64 > 1) take(641, 1, cs.n64[0] + cs.n64[1] * nk * n64);
  if (n128 > 1) take(1281, 1, cs.n128[0] + cs.n128[1] * nk * n128);
  if (M >= 512 && slab_bytes > 0) {
    auto persistent = [&](int code, const Tile& t, const float (&x)[4]) {
      if (N % t.bn != 0) return;
      const int n = over(M, 256) * (N / t.bn), rest = n % cus;
      if (rest == 0) return;
      int S = cus / rest > 8 ? 8 : cus / rest;
      while (S > 1 && nk / S < 4) --S;
      take(code, n < cus ? S : 0, (n / cus) * (t.a + t.b * nk) + x[0] + x[1] * nk / S + (S > 1 ? x[2] + x[3] * (S - 1) : 0.f));
    };
    persistent(1025, cs.tiles[0], cs.p256);
    persistent(769, cs.tiles[1], cs.p128);
  }
  return best;
}

// 128-column tiles of the two-deep ring (else 64): forced, or where they fill the chip
static bool two_deep_wide(int M, int N, int code) {
  if (code == 64 || N % 128 != 0) return false;
  return code == 128 || (M + 127) / 128 * (N / 128) >= 240;
}

// K slices of a forced tile: `sk` of them, or (0) enough for about a block per CU in tiles of the two-deep ring; at least four K-tiles
// each, and no more than the workspace holds
int prefill_slices(int M, int N, int K, int code, int sk, size_t slab_bytes) {
  int nz = sk > 0 ? sk : 1;
  if (sk <= 0 && code < 5000) {
    const int blocks = (M + 127) / 128 * (N / (two_deep_wide(M, N, code) ? 128 : 64));
    if (blocks < 200) nz = min(8, (256 + blocks - 1) / blocks);
  }
  while (nz > 1 && K / 64 / nz < 4) --nz;
  return nz > 1 && ((size_t)nz * M * N + (size_t)nz * M) * 4 > slab_bytes ? 1 : nz;
}

// The cheapest form with `cut` K slices (gemm_prompt_q4.hip compares it)
PrefillForm prefill_form_cut(int M, int N, int K, bool norm, bool rows16, size_t slab_bytes, int cut) {
  return choose_prefill_form(M, N, K, norm, rows16, slab_bytes > 0, slab_bytes, slab_bytes > 0, cut);
}

template <int EPI, int NORM>
bool launch_gemm_w4(const GemmParams& p, int code, int nz, hipStream_t st);

// Returns false for shapes the kernels do not take (the caller keeps the N-split tile
// kernels): K % 64, N % 64, a row gather but of fp32 outputs on four-wave tiles, the gamma-in-registers RMSNorm mode. A forced form that N is no multiple of: false too, but an
// error for the four-wave tiles.
template <int EPI, int NORM>
static bool launch_prefill_epi(const GemmParams& p, int force_bn, int force_sk, size_t slab_bytes, int max_counters, int64_t span,
                               hipStream_t st) {
  constexpr int NTB = 1;  // every epilogue works on self-contained 16-column tiles
  if (p.K % 64 != 0 || p.N % 64 != 0) return false;
  if (p.row_idx != nullptr && (EPI != EPI_F32 || force_bn < 5000 || span >= (1ll << 31))) return false;
  // the four-wave forms address a block's rows of x by 32-bit offsets and fetch them in 16-B pieces
  const bool rows16 = reinterpret_cast<uintptr_t>(p.x) % 16 == 0 && p.lda % 8 == 0 && p.lda < (1 << 20) && p.K < (1 << 20);
  if (force_bn == 0 && force_sk == 0) {
    const PrefillForm f = choose_prefill_form(p.M, p.N, p.K, NORM == 2, rows16, p.slabs != nullptr, slab_bytes, p.counters != nullptr);
    force_bn = f.code;
    force_sk = f.nz;
  }
  const int nz = prefill_slices(p.M, p.N, p.K, force_bn, force_sk, p.slabs != nullptr ? slab_bytes : 0);
  if (force_bn >= 5000) {
    if (!rows16) return false;
    if (!launch_gemm_w4<EPI, NORM>(p, force_bn, nz, st)) throw std::runtime_error("gemm: no such four-wave tile, or none of N");
    if (nz > 1) launch_prefill_reduce<EPI, NORM, 1>(p, nz, st);
    return true;
  }
  if (force_bn == 1024) {  // the 4-phase 256 x 256 kernel
    if (p.N % 256 != 0) return false;
    launch_prefill4_cfg<EPI, NORM, NTB>(p, nz, st);
    return true;
  }
  if (force_bn == 768) {  // on a 256 x 128 tile
    if (p.N % 128 != 0) return false;
    launch_prefill4_cfg<EPI, NORM, NTB, 128>(p, nz, st);
    return true;
  }
  // persistent forms of the 4-phase kernel, K-split tail (force_sk = the tail's K slices); declined -> the tile grid
  if (force_bn == 1025) {
    if (p.N % 256 != 0) return false;
    if (!launch_prefill4sk_cfg<EPI, NORM, NTB, 256>(p, force_sk, max_counters, slab_bytes, st))
      launch_prefill4_cfg<EPI, NORM, NTB>(p, 1, st);
    return true;
  }
  if (force_bn == 769) {
    if (p.N % 128 != 0) return false;
    if (!launch_prefill4sk_cfg<EPI, NORM, NTB, 128>(p, force_sk, max_counters, slab_bytes, st))
      launch_prefill4_cfg<EPI, NORM, NTB, 128>(p, 1, st);
    return true;
  }
  // 128-row tiles over 8 waves on a 4-deep ring, one block per CU
  if (force_bn == 1281) {
    if (p.N % 128 != 0) return false;
    launch_prefill2_cfg<EPI, NORM, NTB, 128, 128, 2, 4, 4>(p, nz, st);
    return true;
  }
  if (force_bn == 641) {
    launch_prefill2_cfg<EPI, NORM, NTB, 128, 64, 4, 2, 4>(p, nz, st);
    return true;
  }
  // Sweeps and tests only: 256 x 128 on a 3-deep ring, 256 x 256 on a 2-deep one, the 128-row tiles above over 4 waves, 64 x 512 and
  // 128 x 320 (with 32-deep stages on 4-deep rings those took 15-30 % longer, warm and cold: profiles/r5_prefill_wide_tiles_sweep.log), and,
  // for any other code, 128 x 128 or 128 x 64 on a 2-deep ring, which waits for the stage it has just asked for and relies on a second block.
  if constexpr (EPI != EPI_GLU) {
    const int width = force_bn == 512 ? 256 : force_bn == 2560 ? 512 : force_bn == 2561 ? 320 : force_bn == 256 || force_bn == 1280 ? 128 : 64;
    if (p.N % width != 0) return false;
    if (force_bn == 256) launch_prefill2_cfg<EPI, NORM, NTB>(p, nz, st);
    else if (force_bn == 512) launch_prefill2_cfg<EPI, NORM, NTB, 256, 256, 4, 2, 2>(p, nz, st);
    else if (force_bn == 1280) launch_prefill2_cfg<EPI, NORM, NTB, 128, 128, 2, 2, 4>(p, nz, st);
    else if (force_bn == 640) launch_prefill2_cfg<EPI, NORM, NTB, 128, 64, 2, 2, 4>(p, nz, st);
    else if (force_bn == 2560) launch_prefill2_cfg<EPI, NORM, NTB, 64, 512, 1, 8, 2>(p, nz, st);
    else if (force_bn == 2561) launch_prefill2_cfg<EPI, NORM, NTB, 128, 320, 2, 4, 2>(p, nz, st);
    else if (two_deep_wide(p.M, p.N, force_bn)) launch_prefill_cfg<128, 128, EPI, NORM, NTB>(p, nz, st);
    else launch_prefill_cfg<128, 64, EPI, NORM, NTB>(p, nz, st);
    return true;
  }
  return false;
}

bool launch_gemm_prefill(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0) return true;
  const int norm = g.norm_w != nullptr ? 1 : (g.rownorm ? 2 : 0);
  if (norm == 1) return false;
  GemmParams p{};
  p.x = g.x; p.lda = g.lda; p.M = g.M; p.row_idx = g.row_idx;
  p.wp = reinterpret_cast<const uint4*>(g.wp); p.N = g.N; p.K = g.K;
  p.norm_w = nullptr; p.eps = g.eps;
  p.bias = g.bias; p.res = g.res; p.ldr = g.ldr;
  p.out = g.out; p.ldo = g.ldo;
  p.splitk = 1;
  p.slabs = g.slabs;
  p.counters = g.counters; p.fault = g.fault;
  p.positions = g.positions; p.slots = g.slots; p.cos_sin = g.cos_sin;
  p.k_cache = g.k_cache; p.v_cache = g.v_cache; p.hq = g.hq; p.hkv = g.hkv; p.bs = g.bs;
  if (g.act != 0) set_glu(p, GluAct{g.act, g.limit, g.alpha});
  p.dbg_ts = g.dbg_ts;
  const int fb = g.ntb;      // reused as the forced tile width (0 = heuristic, 64 / 128)
  const int fs = g.splitk;   // forced K slices (0 = heuristic)
#define VG_PF(E)                                                                                         \
  return norm == 2 ? launch_prefill_epi<E, 2>(p, fb, fs, g.slab_bytes, g.max_counters, g.x_span, st)               \
                   : launch_prefill_epi<E, 0>(p, fb, fs, g.slab_bytes, g.max_counters, g.x_span, st)
  if (g.act != 0) return launch_prefill_epi<EPI_GLU, 0>(p, fb, fs, g.slab_bytes, g.max_counters, g.x_span, st);
  switch (g.epi) {
    case EPI_SILU: VG_PF(EPI_SILU);
    case EPI_QKV: VG_PF(EPI_QKV);
    case EPI_F32: VG_PF(EPI_F32);
    default: VG_PF(EPI_BF16);
  }
#undef VG_PF
}

}  // namespace vgate
