// Prompt GEMM on four waves, one per SIMD: each computes a quarter (2 x 2) of the block tile, MT x NT MFMA tiles of 16 x 16, so a block
// is 32 MT rows x 32 NT columns and the sizes between the powers of two come for the asking.
//
// What bounds it. A K-tile of 64 asks a CU for (BM + BN) x 128 B from L2 (25 to 30 B per clock and CU with all of them at it: 64 x 64
// tiles 0.25 us a K-tile for the loads alone, 0.31 in all), for (MT + NT) x 16 KiB of fragment reads (108 B per clock) and for BM x BN / 32
// matrix cycles; from 160 x 256 on the matrix cores bound it, at the clock that their power leaves (1.5 to 2.1 GHz on random data: a K-tile
// of 256 x 256 1.1 to 1.4 us at best, 1.6 here as in the four-phase kernel of gemm_prefill.hip). So:
//   * a wave reads its fragments once per k-step into registers, 32 B of LDS per MFMA where eight waves of half the size read 48;
//   * the reads of a k-step are under way during the MFMAs of the one before (two register sets), the DMA of a K-tile during the NS - 1
//     before it, and one barrier per K-tile stands between its two k-steps, where every operand of the second is in registers already;
//   * accumulators stay in AGPRs (mfma_acc), addresses in SGPRs (blds16): the loop is MFMA, ds_read and DMA only.
// us, eight-wave forms -> these (MI355X, cold weights): 64 x 64 tiles 2048 x 1536 at 448 rows 17.1 -> 12.6, 1536 x 1536 at 256 16.6 -> 12.5,
// 1024 x 4096 at 1024 32.2 -> 24.0; 160 x 256 17920 x 1536 at 448 46.8 -> 38.8, 4352 x 1024 at 2048 36.6 -> 30.3; 192 x 128 17920 x 1536 at
// 1024 87 -> 80. As 256 x 256 tiles it is no faster than the four-phase kernel (28672 x 4096 at 2048 rows 445, 449), which keeps those.
#pragma once
#include <type_traits>

#include "gemm_epilogue.h"
#include "lds_rows.h"

namespace vgate {

// The epilogue of a wave's MT x NT tiles of a prompt GEMM (rows m0 + 16 b, tiles nt0 + a; value(a, b): the tile's accumulator, row scale
// applied): epilogue()'s results, with what does not depend on the tile loaded, and divided, once per row. Tile by tile the loads of
// positions, rotations, slots and residuals cannot pass the stores before them (they may alias), and every tile waits for memory:
// Llama-3-8B prompt of 2048 tokens, step 3538 -> 3491 us.
template <int NT, int MT, int EPI, typename V>
__device__ __forceinline__ void prompt_epilogue(const GemmParams& p, int m0, int nt0, int lane, V value) {
  const int nsub = 4 * (lane >> 4);
  if constexpr (EPI == EPI_QKV && 8 % NT == 0) {  // the wave's tiles lie in one head
    const int head = __builtin_amdgcn_readfirstlane(nt0 >> 3);
    const bool rotated = head < p.hq + p.hkv, upper = nsub >= 8;
    const int d0 = qkv_rot(nt0, nsub), dcol = (upper ? 64 : 0) + d0;
    uint2 bias[NT];
    int pos[MT], slot[MT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
      bias[a] = p.bias ? *reinterpret_cast<const uint2*>(p.bias + qkv_col(nt0 + a, nsub)) : make_uint2(0, 0);
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int mm = min(m0 + b * 16 + (lane & 15), p.M - 1);
      pos[b] = rotated ? p.positions[mm] : 0;
      slot[b] = p.slots[mm];
    }
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int m = m0 + b * 16 + (lane & 15);
      float4 cs[NT], sn[NT];
      if (rotated) {
        const float* cp = p.cos_sin + (size_t)pos[b] * 128 + d0;
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          cs[a] = *reinterpret_cast<const float4*>(cp + 8 * a);
          sn[a] = *reinterpret_cast<const float4*>(cp + 64 + 8 * a);
        }
      }
      bf16_t* dst;
      if (head < p.hq) {
        dst = reinterpret_cast<bf16_t*>(p.out) + (size_t)m * p.ldo + head * 128 + dcol;
      } else {
        const int blk = slot[b] / p.bs, kh = rotated ? head - p.hq : head - p.hq - p.hkv;
        dst = (rotated ? p.k_cache : p.v_cache) + (((size_t)blk * p.hkv + kh) * p.bs + (slot[b] - blk * p.bs)) * 128 + dcol;
      }
      const bool store = m < p.M && (head < p.hq || slot[b] >= 0);
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const f32x4 v = value(a, b);
        const float bb[4] = {bf_lo(bias[a].x), bf_hi(bias[a].x), bf_lo(bias[a].y), bf_hi(bias[a].y)};
        float x[4], xp[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = bf2f(f2bf(v[i] + bb[i]));  // qkv is bf16 in the reference: round before rotating
        if (rotated) {
          const float cc[4] = {cs[a].x, cs[a].y, cs[a].z, cs[a].w}, sc[4] = {sn[a].x, sn[a].y, sn[a].z, sn[a].w};
#pragma unroll
          for (int i = 0; i < 4; ++i) xp[i] = xor32(x[i]);  // the partner column's value (all 64 lanes active)
#pragma unroll
          for (int i = 0; i < 4; ++i) x[i] = upper ? x[i] * cc[i] + xp[i] * sc[i] : x[i] * cc[i] - xp[i] * sc[i];
        }
        if (store) *reinterpret_cast<uint2*>(dst + 8 * a) = make_uint2(pack_bf2(x[0], x[1]), pack_bf2(x[2], x[3]));
      }
    }
  } else if constexpr (EPI == EPI_BF16 || EPI == EPI_F32) {
    uint2 bias[NT], res[2][NT];
    auto load_res = [&](int b) {
      const bf16_t* r = p.res + (size_t)min(m0 + b * 16 + (lane & 15), p.M - 1) * p.ldr + nt0 * 16 + nsub;
#pragma unroll
      for (int a = 0; a < NT; ++a) res[b & 1][a] = *reinterpret_cast<const uint2*>(r + 16 * a);
    };
    if (p.bias) {
#pragma unroll
      for (int a = 0; a < NT; ++a) bias[a] = *reinterpret_cast<const uint2*>(p.bias + (nt0 + a) * 16 + nsub);
    }
    if (EPI == EPI_BF16 && p.res) load_res(0);
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      if (EPI == EPI_BF16 && b + 1 < MT && p.res) load_res(b + 1);  // (rows of its own: out may be the residual)
      const int m = m0 + b * 16 + (lane & 15);
      if (m < p.M) {
#pragma unroll
        for (int a = 0; a < NT; ++a) {
          const f32x4 v[1] = {value(a, b)};
          EpiPre<1> e;
          e.b0 = bias[a];
          e.r0 = res[b & 1][a];
          epilogue<1, EPI, true>(p, v, m, nt0 + a, nsub, e, true);
        }
      }
    }
  } else {
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int m = m0 + b * 16 + (lane & 15);
#pragma unroll
      for (int a = 0; a < NT; ++a) {
        const f32x4 v[1] = {value(a, b)};
        epilogue<1, EPI, false>(p, v, m, nt0 + a, nsub, EpiPre<1>{}, m < p.M);
      }
    }
  }
}

template <int MT, int NT>
struct W4 {  // geometry: block (32 MT) rows x (32 NT) columns, stages of 64 k
  static constexpr int BM = 32 * MT, BN = 32 * NT;
  static constexpr int PPW = MT + NT;             // 1 KiB pieces per wave and stage
  static constexpr int STAGE = 4 * PPW * 1024;
};

// NS: stages in LDS. K-split (grid.y), epilogues and the order of the blocks as in gemm_prefill.hip.
template <int MT, int NT, int NS, int EPI, int NORM>
__global__ __launch_bounds__(256, 1) void gemm_w4_kernel(GemmParams p) {
  using G = W4<MT, NT>;
  constexpr int PPW = G::PPW, STAGE = G::STAGE, WPC = NT;  // W pieces of a wave: NT (NT / 2 tiles x 2 k-steps)
  constexpr int XB = 4 * NT * 1024;                        // x tiles of a stage lie behind its W tiles
  static_assert(NT % 2 == 0 && (MT * NT) % 4 == 0 && NS >= 2 && (NS - 1) * PPW < 64, "pieces per wave, groups of four MFMAs, vmcnt");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TLScope tl_scope(p.dbg_ts);
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const int KT = p.K >> 5, nk_all = p.K >> 6;
  const int z = blockIdx.y, nz = gridDim.y;
  const int kst0 = (nk_all * z) / nz, nk = (nk_all * (z + 1)) / nz - kst0;
  const int mblocks = (p.M + G::BM - 1) / G::BM;
  const int nwg = gridDim.x, orig = blockIdx.x, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int wgid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  // groups of up to 8 row blocks, inside a group rows fastest: the blocks that run together on an XCD share few panels of both operands
  // (rows fastest over all of them, 64 x 64 tiles: 1024 x 4096 at 2048 rows 44.5 -> 36.2 us; a group of 2, 4 or 8 is the same)
  const int per = 8 * (p.N / G::BN), grp = wgid / per, in = wgid - grp * per, gm = min(8, mblocks - 8 * grp);
  const int m0 = (8 * grp + in % gm) * G::BM;
  const int nt_blk = (in / gm) * (2 * NT);
  const u32x4 wrs = rsrc_words(p.wp + ((size_t)nt_blk * KT + 2 * kst0) * 64);
  const bool gather = EPI == EPI_F32 && p.row_idx != nullptr;   // (LM heads; every row within 2 GiB of the first: the launcher)
  const u32x4 xrs = rsrc_words(p.x + (gather ? 0 : (size_t)m0 * p.lda) + kst0 * 64);
  const uint32_t wvo = lane * 16;
  uint32_t xvo[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int g = wid * MT + i;
    const int row = x_piece_row(m0 + (g >> 1) * 16, g & 1, lane, p.M);
    xvo[i] = (uint32_t)(gather ? p.row_idx[row] : row - m0) * (uint32_t)p.lda * 2u + (uint32_t)x_piece_col(g & 1, lane) * 2u;
  }
  const uint32_t lds0 = lds_addr_of(smem);
  const uint32_t wrow = (uint32_t)KT * 1024u, wso0 = (uint32_t)wid * (NT / 2) * wrow;
  // piece i of this wave's share of `stage` into `buf`
  auto issue_piece = [&](int i, int st, int buf) {
    if (i < WPC) blds16(wrs, wvo, wso0 + (uint32_t)(i >> 1) * wrow + (uint32_t)(2 * st + (i & 1)) * 1024u,
                        lds0 + buf * STAGE + (uint32_t)(wid * NT + i) * 1024u);
    else blds16(xrs, xvo[i - WPC], (uint32_t)st * 128u, lds0 + buf * STAGE + XB + (uint32_t)(wid * MT + i - WPC) * 1024u);
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[a][b]));  // (written here, well before the first mfma_acc)
    }
  float ss[MT];
#pragma unroll
  for (int b = 0; b < MT; ++b) ss[b] = 0.f;
  uint4 wf[2][NT], xf[2][MT];
  const int wlo = lane * 16 + wn * NT * 2048, xlo[2] = {XB + wm * MT * 2048 + x_frag_off(0, lane), XB + wm * MT * 2048 + x_frag_off(1, lane)};
  // fragment read rd (0: W tile 0, 1 .. MT: x, then the other W tiles: the order in which a phase needs them)
  auto read_frag = [&](int rd, int ks, const char* sb) {
    if (rd == 0) wf[ks][0] = *reinterpret_cast<const uint4*>(sb + wlo + ks * 1024);
    else if (rd <= MT) xf[ks][rd - 1] = *reinterpret_cast<const uint4*>(sb + xlo[ks] + (rd - 1) * 2048);
    else wf[ks][rd - MT] = *reinterpret_cast<const uint4*>(sb + wlo + (rd - MT) * 2048 + ks * 1024);
  };
  constexpr int GR = MT * NT / 4, RD = MT + NT;
  constexpr int HG = GR > 1 ? GR / 2 : 1, RPG = (RD + HG - 1) / HG;  // reads per group: done by the middle of the phase
  // one phase: the MFMAs of k-step ks in groups of four, between them the reads of the other k-step (from sb) and, if `dma`, the next
  // stage's pieces
  auto phase = [&](auto ksc, const char* sb, auto dmac, int st, int buf) {
    constexpr int ks = decltype(ksc)::value, dma = decltype(dmac)::value;
#pragma unroll
    for (int g = 0; g < GR; ++g) {
#pragma unroll
      for (int u = 0; u < RPG; ++u)
        if (g * RPG + u < RD) read_frag(g * RPG + u, ks ^ 1, sb);
      if constexpr (dma) {
#pragma unroll
        for (int i = (g * PPW) / GR; i < ((g + 1) * PPW) / GR; ++i) issue_piece(i, st, buf);
      }
#pragma unroll
      for (int e = 4 * g; e < 4 * g + 4; ++e) {
        const int a = e / MT, b = e % MT;
        if constexpr (NORM == 2)
          if (a == NT / 2) ss[b] = sumsq8(xf[ks][b], ss[b]);
        mfma_acc(acc[a][b], wf[ks][a], xf[ks][b]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
#pragma unroll
  for (int s0 = 0; s0 < NS; ++s0)
#pragma unroll
    for (int i = 0; i < PPW; ++i) issue_piece(i, s0 < nk ? s0 : nk - 1, s0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * PPW) : "memory");
#pragma unroll
  for (int rd = 0; rd < RD; ++rd) read_frag(rd, 0, smem);
  int buf = 0;
  for (int t = 0; t < nk; ++t) {
    const char* sb = smem + buf * STAGE;
    const int nb = buf + 1 == NS ? 0 : buf + 1;
    phase(C0{}, sb, C0{}, 0, 0);
    // this stage is read (its second k-step is in registers), the next one has landed: both for every wave
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * PPW) : "memory");
    const int st = t + NS < nk ? t + NS : nk - 1;  // past the end: clamped duplicates, never used
    phase(C1{}, smem + nb * STAGE, C1{}, st, buf);
    buf = nb;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");  // the trailing duplicates
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) asm volatile("" : "+a"(acc[a][b]));
  if (nz > 1) {  // fp32 partial of this K slice, as the other forms leave it for prefill_reduce_kernel
    float* part = p.slabs + (size_t)z * p.M * p.N;
    float* ssq = p.slabs + (size_t)nz * p.M * p.N + (size_t)z * p.M;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int m = m0 + (wm * MT + b) * 16 + (lane & 15);
      float s2 = 0.f;
      if constexpr (NORM == 2) {
        s2 = ss[b];
        s2 += xor16(s2);
        s2 += xor32(s2);
      }
      if (m < p.M) {
        if (NORM == 2 && wn == 0 && nt_blk == 0 && lane < 16) ssq[m] = s2;
#pragma unroll
        for (int a = 0; a < NT; ++a)
          __builtin_nontemporal_store(acc[a][b], reinterpret_cast<f32x4*>(part + (size_t)m * p.N + (nt_blk + wn * NT + a) * 16 + 4 * (lane >> 4)));
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
  prompt_epilogue<NT, MT, EPI>(p, m0 + wm * MT * 16, nt_blk + wn * NT, lane, [&](int a, int b) { return NORM == 2 ? acc[a][b] * sc[b] : acc[a][b]; });
}

}  // namespace vgate
