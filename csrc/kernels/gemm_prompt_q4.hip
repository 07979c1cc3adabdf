// Prompt GEMM on int4 weights (AWQ, groups of 128): the weights are unpacked between LDS and the matrix cores, so a step reads them at
// 4 bits and no bf16 copy is written and read back. Every fragment holds the very bf16 values of that copy ((v s - s z) gamma, rounded once),
// and products and squares are summed in the order of the bf16 forms: the bits are theirs.
//
// As gemm_w4_kernel (gemm_prompt.h): operands of a k-step are read (here: and unpacked) during the MFMAs of the one before, stages come by
// LDS-DMA. The waves stand side by side over the columns, so that each fragment of W is unpacked by one wave of the block only.
// What bounds it is the issue of vector instructions. One wave on a SIMD issues one every 5 to 6 cycles (a conversion every 8) whatever else
// is ready; two or more take 4.3 each between MFMAs, which take 8 of issue and 16 of the matrix core. So tiles are made for two waves to a SIMD
// and more, eight in a block or two to four blocks of four or eight on a CU (stages of 128 k, two or three of them as LDS allows); one is left
// where a launch has too few blocks of four waves, in tile 410 with a norm in front of slices of more than 2900 (their gamma takes the second
// block's LDS) and in tile 1620. Weights turn into floats without conversions (unpack()); gamma is widened once per block and not once per
// wave and k-step. Per fragment 17 vector instructions, 25
// with gamma, against MT MFMAs. LDS is next: an x fragment (8 cycles) serves NT MFMAs.
// us, four waves with 23 and 31 instructions -> these (MI355X, cold weights, the same slices): 256 rows, 17920 x 1536 with a norm 35.1 -> 29.3,
// 1536 x 8960 in 8 slices 27.3 -> 21.8, 1536 x 1536 11.4 -> 10.1; 448 rows, 17920 x 1536 55.9 -> 45.4, 1536 x 8960 31.6 -> 27.4; 96 rows 23.8 ->
// 18.9 and 16.0 -> 15.5; a step of 256 rows through six layers of 1536 / 8960 694 -> 645.
#include "gemm_prompt.h"

namespace vgate {

template <int NW, int MT, int NT, bool RING>
struct Q4 {  // geometry: NW waves side by side, each 16 MT rows x 16 NT columns; stages of 128 k (one group)
  static constexpr int BM = 16 * MT, BN = 16 * NW * NT;
  static constexpr int XB = BN * 64, SB = XB + BM * 256;  // W | x (two 64-k halves) | scales, zeros, RING: gamma: 1 KiB each
  static constexpr int STAGE = SB + (RING ? 3072 : 2048);
  static constexpr int XPW = 4 * MT / NW, PPW = XPW + NT + 1;  // x pieces and all DMA of a wave and stage
};

// RING: gamma comes with the stages, bf16, and is widened per wave and k-step; else the slice's stands in LDS as fp32.
template <int NW, int MT, int NT, int NS, int EPI, bool NORM, bool RING>
__global__ __launch_bounds__(64 * NW, NW / 4) void gemm_q4_prompt_kernel(GemmParams p) {
  using G = Q4<NW, MT, NT, RING>;
  static_assert(!RING || (NORM && NW == 4), "two waves' small pieces are gamma");
  constexpr int PPW = G::PPW, XPW = G::XPW, STAGE = G::STAGE;
  static_assert(NS * STAGE <= 160 * 1024 && XPW * NW == 4 * MT, "LDS; x in equal shares");
  static_assert(NS >= 2 && (NS - 1) * PPW < 64 && (G::BN & (G::BN - 1)) == 0 && G::BN <= 512, "vmcnt; the block's scales repeat in 1 KiB");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  TLScope tl_scope(p.dbg_ts);
  const int lane = threadIdx.x & 63, quad = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int KQ = p.K >> 7;
  // K slices in tiles of 64 k, as the bf16 forms cut them: a slice can begin or end inside a group, whose other half then counts as zeros
  const int z = blockIdx.y, nz = gridDim.y, kt0 = (2 * KQ * z) / nz, kt1 = (2 * KQ * (z + 1)) / nz;
  const int q0 = kt0 >> 1, nk = ((kt1 + 1) >> 1) - q0;
  const int mblocks = (p.M + G::BM - 1) / G::BM;
  const int nwg = gridDim.x, orig = blockIdx.x, xcd = orig & 7, q = nwg >> 3, r = nwg & 7;
  const int wgid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (orig >> 3);
  const int per = 8 * (p.N / G::BN), grp = wgid / per, in = wgid - grp * per, gm = min(8, mblocks - 8 * grp);
  const int m0 = (8 * grp + in % gm) * G::BM;
  const int n0 = (in / gm) * G::BN, nt0 = n0 / 16 + wid * NT;  // the wave's first column tile
  const u32x4 wrs = rsrc_words(p.wp + ((size_t)(n0 / 16) * KQ + q0) * 64);
  const u32x4 xrs = rsrc_words(p.x + (size_t)m0 * p.lda + q0 * 128);
  // the wave's small piece: the group's scales or zeros of the block's columns or its gamma, asked for again until the 1 KiB is full
  const int kind = RING ? min(wid, 2) : wid & 1;
  const bf16_t* small = kind == 0 ? p.scales : kind == 1 ? p.zeros : p.norm_w;
  const u32x4 srs = rsrc_words(small + (kind < 2 ? (size_t)q0 * p.N + n0 : (size_t)q0 * 128));
  const uint32_t sstep = kind < 2 ? (uint32_t)p.N * 2u : 256u;
  const uint32_t wvo = lane * 16, svo = (uint32_t)(lane * 16) & (kind < 2 ? 2u * G::BN - 1u : 255u);
  uint32_t xvo[XPW];  // pieces of 8 rows x 64 k: tile (piece >> 2), k half (piece >> 1) & 1, row half piece & 1
#pragma unroll
  for (int i = 0; i < XPW; ++i) {
    const int g = wid * XPW + i;
    xvo[i] = (uint32_t)(x_piece_row(m0 + (g >> 2) * 16, g & 1, lane, p.M) - m0) * (uint32_t)p.lda * 2u + (uint32_t)x_piece_col(g & 1, lane) * 2u +
             (uint32_t)((g >> 1) & 1) * 128u;
  }
  const uint32_t lds0 = lds_addr_of(smem);
  const uint32_t wrow = (uint32_t)KQ * 1024u;
  auto issue_piece = [&](int i, int st, int buf) {
    const uint32_t base = lds0 + buf * STAGE;
    if (i < NT) blds16(wrs, wvo, (uint32_t)(wid * NT + i) * wrow + (uint32_t)st * 1024u, base + (uint32_t)(wid * NT + i) * 1024u);
    else if (i < NT + XPW) blds16(xrs, xvo[i - NT], (uint32_t)st * 256u, base + G::XB + (uint32_t)(wid * XPW + i - NT) * 1024u);
    else blds16(srs, svo, (uint32_t)st * sstep, base + G::SB + kind * 1024u);
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[a][b]));  // (written here, well before the first mfma_acc)
    }
  // wave w sums the squares of the row tiles w, w + NW, ...: a row in the order of K, as the bf16 forms do. It reads them again: which of the
  // fragments in registers are its own would be a branch per k-step, around which the accumulators lose their place (5 to 7 times as long)
  constexpr int SQ = NORM ? (MT + NW - 1) / NW : 1;
  float ss[SQ];
  int so[SQ];
#pragma unroll
  for (int i = 0; i < SQ; ++i) {
    ss[i] = 0.f;
    so[i] = min(wid + NW * i, MT - 1) * 4096;
  }
  uint4 wf[2][NT], xf[2][MT], wq[NT], sq[2][SQ];
  float sc[NT], sc4[NT], zs[NT];
  float4 gam[2];
  const int xlo[2] = {G::XB + x_frag_off(0, lane), G::XB + x_frag_off(1, lane)};
  auto read_stage = [&](const char* sb) {  // the group's packed weights and scales
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      wq[a] = *reinterpret_cast<const uint4*>(sb + (wid * NT + a) * 1024 + lane * 16);
      const float s = bf2f(*reinterpret_cast<const bf16_t*>(sb + G::SB + ((wid * NT + a) * 16 + (lane & 15)) * 2));
      sc[a] = s * 0x1p24f;
      sc4[a] = s * 0x1p20f;
      zs[a] = bf2f(*reinterpret_cast<const bf16_t*>(sb + G::SB + 1024 + ((wid * NT + a) * 16 + (lane & 15)) * 2));
    }
  };
  const char* gbase = smem + NS * STAGE + quad * 32;  // gamma of the slice, fp32
  auto read_gamma = [&](int u, int t, const char* sb) {
    if constexpr (RING) {
      float g[8];
      unpack8(*reinterpret_cast<const uint4*>(sb + G::SB + 2048 + u * 64 + quad * 16), g);
      gam[0] = make_float4(g[0], g[1], g[2], g[3]);
      gam[1] = make_float4(g[4], g[5], g[6], g[7]);
    } else if constexpr (NORM) {
      gam[0] = *reinterpret_cast<const float4*>(gbase + t * 512 + u * 128);
      gam[1] = *reinterpret_cast<const float4*>(gbase + t * 512 + u * 128 + 16);
    }
  };
  // half h of the wave's fragment of tile a at k-step u: the bf16 that the unpacked copy of the matrix would hold. The low nibbles of a
  // word's bytes are elements 0 4 1 5, the high ones 2 6 3 7: two of them, 16 bits apart, are a pair of f16 subnormals v 2^-24 (the high
  // ones v 2^-20), exact, which v_fma_mix_f32 takes as they stand: v s - s z in one rounding without a conversion of v. (2^24 s has to be
  // finite: a matrix with a scale of 2^104 or more goes by way of its copy, Linear.prompt_scales of vgate/ops.)
  auto unpack = [&](int a, int h, int u) {
    const uint32_t w = u == 0 ? wq[a].x : u == 1 ? wq[a].y : u == 2 ? wq[a].z : wq[a].w;
    const uint32_t lo = w & (h ? 0x00F000F0u : 0x000F000Fu), hi = (w >> 8) & (h ? 0x00F000F0u : 0x000F000Fu);
    const float s = h ? sc4[a] : sc[a];
    float f[4];
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[1,0,0]" : "=v"(f[0]) : "v"(lo), "v"(s), "v"(zs[a]));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(f[1]) : "v"(lo), "v"(s), "v"(zs[a]));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[1,0,0]" : "=v"(f[2]) : "v"(hi), "v"(s), "v"(zs[a]));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(f[3]) : "v"(hi), "v"(s), "v"(zs[a]));
    if constexpr (NORM) {
      f[0] *= h ? gam[0].z : gam[0].x;
      f[1] *= h ? gam[0].w : gam[0].y;
      f[2] *= h ? gam[1].z : gam[1].x;
      f[3] *= h ? gam[1].w : gam[1].y;
    }
    uint4& o = wf[u & 1][a];
    (h ? o.y : o.x) = pack_bf2(f[0], f[1]);
    (h ? o.w : o.z) = pack_bf2(f[2], f[3]);
  };
  auto read_x = [&](int b, int u, const char* sb) {
    xf[u & 1][b] = *reinterpret_cast<const uint4*>(sb + xlo[u & 1] + b * 4096 + (u >> 1) * 2048);
    if constexpr (NORM)
      if (b < SQ) sq[u & 1][b] = *reinterpret_cast<const uint4*>(sb + xlo[u & 1] + so[b] + (u >> 1) * 2048);
  };
  // zeros in place of a stage's k half that belongs to the slice before or after (once in a slice at either end; no wave is reading it)
  auto clear = [&](char* sb, int half) {
    for (int e = threadIdx.x; e < MT * 128; e += 64 * NW)
      *reinterpret_cast<uint4*>(sb + G::XB + (e >> 7) * 4096 + half * 2048 + (e & 127) * 16) = make_uint4(0, 0, 0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  constexpr int U = 2 * NT;  // halves of fragments of a k-step to unpack
  // the MFMAs of k-step u, a row tile at a time; between them the next k-step is read and unpacked and, at the last, the next stage asked for
  auto phase = [&](auto uc, const char* sb, int t, int st, int buf) {
    constexpr int u = decltype(uc)::value, v = (u + 1) & 3;
    // (an MFMA reads what the VALU wrote two wait states before at the soonest, and the compiler does not see that mfma_acc() is one)
#pragma unroll
    for (int a = 0; a < NT; ++a) {
      u32x4 f = __builtin_bit_cast(u32x4, wf[u & 1][a]);
      asm volatile("s_nop 1" : "+v"(f));
      wf[u & 1][a] = __builtin_bit_cast(uint4, f);
    }
    if constexpr (u == 3) read_stage(sb);
    read_gamma(v, t, sb);
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      if constexpr (NORM)
        if (b < SQ) ss[b] = sumsq8(sq[u & 1][b], ss[b]);
      read_x(b, v, sb);
      if constexpr (u == 3) {
#pragma unroll
        for (int i = (b * PPW) / MT; i < ((b + 1) * PPW) / MT; ++i) issue_piece(i, st, buf);
      }
#pragma unroll
      for (int e = (b * U) / MT; e < ((b + 1) * U) / MT; ++e) unpack(e >> 1, e & 1, v);
#pragma unroll
      for (int a = 0; a < NT; ++a) mfma_acc(acc[a][b], wf[u & 1][a], xf[u & 1][b]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;
  // gamma of the slice: bf16 by DMA into the second half of its place (asked for first: it has landed when the first stage has), widened there
  if constexpr (NORM && !RING) {
    u32x4 grs = rsrc_words(p.norm_w + (size_t)q0 * 128);
    grs[2] = (uint32_t)nk * 256u;
    for (int i = wid; i < (nk + 3) >> 2; i += NW) blds16(grs, wvo, (uint32_t)i * 1024u, lds0 + NS * STAGE + ((nk + 3) >> 2) * 1024 + i * 1024u);
  }
#pragma unroll
  for (int s0 = 0; s0 < NS; ++s0)
#pragma unroll
    for (int i = 0; i < PPW; ++i) issue_piece(i, s0 < nk ? s0 : nk - 1, s0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * PPW) : "memory");
  if constexpr (NORM && !RING) {
    const bf16_t* raw = reinterpret_cast<const bf16_t*>(smem + NS * STAGE + ((nk + 3) >> 2) * 1024);
    float* wide = reinterpret_cast<float*>(smem + NS * STAGE);
    // (in place, from the front: a round of 64 NW elements is read by all before it is written, and lies behind what the next one reads)
    for (int e0 = 0; e0 < nk * 128; e0 += 64 * NW) {
      const int e = e0 + threadIdx.x;
      const float g = e < nk * 128 ? bf2f(raw[e]) : 0.f;
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (e < nk * 128) wide[e] = g;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  if (kt0 & 1) clear(smem, 0);
  read_stage(smem);
  read_gamma(0, 0, smem);
#pragma unroll
  for (int b = 0; b < MT; ++b) read_x(b, 0, smem);
#pragma unroll
  for (int e = 0; e < U; ++e) unpack(e >> 1, e & 1, 0);
  int buf = 0;
  for (int t = 0; t < nk; ++t) {
    char* sb = smem + buf * STAGE;
    const int nb = buf + 1 == NS ? 0 : buf + 1;
    if (t == nk - 1 && (kt1 & 1) != 0) clear(sb, 1);
    phase(C0{}, sb, t, 0, 0);
    phase(C1{}, sb, t, 0, 0);
    phase(C2{}, sb, t, 0, 0);
    // this stage is read (its last k-step is in registers), the next one has landed: both for every wave
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * PPW) : "memory");
    phase(C3{}, smem + nb * STAGE, min(t + 1, nk - 1), t + NS < nk ? t + NS : nk - 1, buf);  // past the end: clamped duplicates, never used
    buf = nb;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");  // the trailing duplicates
#pragma unroll
  for (int a = 0; a < NT; ++a)
#pragma unroll
    for (int b = 0; b < MT; ++b) asm volatile("" : "+a"(acc[a][b]));
  float* rows = reinterpret_cast<float*>(smem);  // sums of squares
  if constexpr (NORM) {
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      float s2 = ss[b / NW];
      s2 += xor16(s2);
      s2 += xor32(s2);
      if (wid == b % NW && lane < 16) rows[b * 16 + lane] = s2;
    }
    __syncthreads();
  }
  float scale[MT], s2[MT];
#pragma unroll
  for (int b = 0; b < MT; ++b) {
    scale[b] = 1.f;
    s2[b] = 0.f;
    if constexpr (NORM) {
      s2[b] = rows[b * 16 + (lane & 15)];
      scale[b] = rsqrtf(s2[b] / (float)p.K + p.eps);
    }
  }
  if (nz > 1) {
    float* part = p.slabs + (size_t)z * p.M * p.N;
    float* ssq = p.slabs + (size_t)nz * p.M * p.N + (size_t)z * p.M;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int m = m0 + b * 16 + (lane & 15);
      if (m < p.M) {
        if (NORM && wid == 0 && n0 == 0 && lane < 16) ssq[m] = s2[b];
#pragma unroll
        for (int a = 0; a < NT; ++a)
          __builtin_nontemporal_store(acc[a][b], reinterpret_cast<f32x4*>(part + (size_t)m * p.N + (nt0 + a) * 16 + 4 * quad));
      }
    }
    return;
  }
  prompt_epilogue<NT, MT, EPI>(p, m0, nt0, lane, [&](int a, int b) { return NORM ? acc[a][b] * scale[b] : acc[a][b]; });
}

// LDS of a slice's gamma: fp32, whole KiB of its bf16 values twice over
static int q4_gamma_lds(int K, int nz) { return (((K >> 6) + nz - 1) / nz + 2) / 2 * 512 + 2048; }

template <int EPI, int NORM, int NTB>
void launch_prefill_reduce(const GemmParams& p, int nz, hipStream_t st);

template <int NW, int MT, int NT, int NS, int EPI, bool NORM, bool RING = false>
static bool launch_q4_one(const GemmParams& p, int nz, hipStream_t st) {
  using G = Q4<NW, MT, NT, RING>;
  const int lds = NS * G::STAGE + (NORM && !RING ? q4_gamma_lds(p.K, nz) : 0);
  if (p.N % G::BN != 0 || lds > 160 * 1024) return false;
  const int blocks = ((p.M + G::BM - 1) / G::BM) * (p.N / G::BN);
  GemmParams q = p;
  if (q.dbg_ts == nullptr) q.dbg_ts = tl_take("gemm_q4_prompt", blocks * nz);
  auto kern = gemm_q4_prompt_kernel<NW, MT, NT, NS, EPI, NORM, RING>;
  static bool attr = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
  }();
  (void)attr;
  hipLaunchKernelGGL(kern, dim3(blocks, nz), dim3(64 * NW), lds, st, q);
  if (nz > 1) launch_prefill_reduce<EPI, NORM ? 2 : 0, 1>(p, nz, st);
  return true;
}

template <int EPI, bool NORM>
static bool launch_q4_epi(const GemmParams& p, int code, int nz, hipStream_t st) {
  switch (code) {
#define VG_Q4(C, NW, MT, NT, NS) case C: return launch_q4_one<NW, MT, NT, NS, EPI, NORM>(p, nz, st)
    VG_Q4(410, 4, 4, 1, 3);
    VG_Q4(412, 4, 4, 1, 2);
    VG_Q4(422, 8, 4, 1, 2);
    VG_Q4(610, 4, 6, 1, 2);
    VG_Q4(620, 8, 6, 1, 2);
    VG_Q4(640, 8, 6, 2, 3);
    VG_Q4(820, 8, 8, 1, 3);
    VG_Q4(1020, 8, 10, 1, 3);
    // four waves: eight would take a column tile each, and LDS 32 cycles of x fragments for 16 of the matrix cores. Long slices
    // leave no room for their gamma, which then comes with the stages (28672 x 4096 at 256 rows 79 us, the next best tile 86; where both fit
    // 0.5 % slower)
    case 1620: return launch_q4_one<4, 16, 2, 2, EPI, NORM>(p, nz, st) || (NORM && launch_q4_one<4, 16, 2, 2, EPI, NORM, NORM>(p, nz, st));
#undef VG_Q4
  }
  return false;
}

// Costs (us) as in choose_prefill_form() of gemm_prefill.hip, fitted to 15 shapes (N 512 .. 28672, K 1024 .. 14336) x 10 row counts 65 ..
// 2048 on cold weights; K-tiles of 128, rounds of as many blocks to a CU as their stages leave room for. Unpacking is repeated by every row
// of blocks, so from some row count on a bf16 copy (2.2 us + 0.56 a million weights) and the bf16 kernels are ahead. Given the slices, the
// choice takes 1.004 of the best tile's time (geometric mean). The copy's estimate is taken at 0.87: measured over estimated, medians of 720
// points (18 shapes x 20 row counts, with a norm and without), 0.80 to 0.93 by form, 0.95 for 256 x 256 tiles in several slices (0.87 there took the
// copy where these tiles are 5 to 8 % ahead: 4096 x 14336 at 768 rows 126, 117); the four-wave forms in one slice at 0.82, since the tiles' own
// estimates are up to 15 % short for many rounds (5120 x 13824 at 2048 rows 323, the copy 270). Over those points the choice takes 1.007 of the
// best form's time.
Q4Form q4_prompt_form(int M, int N, int K, bool norm, bool rows16, bool group128, size_t slab_bytes, int code, int sk) {
  struct Tile {
    int code, bm, bn, stages;
    struct {
      float e, a, b, g, c, d, w, o;
    } cost[2];  // plain, with a norm in front
  };
  static constexpr Tile tiles[] = {
      {410, 64, 64, 3, {{3.09f, 0.61f, 0.181f, 0.285f, 1.84f, 0.675f, 0.026f, 0.466f}, {3.43f, 0.809f, 0.288f, 0.371f, 2.8f, 0.515f, 0.031f, 0.467f}}},
      {412, 64, 64, 2, {{2.65f, 0.f, 0.122f, 0.431f, 2.26f, 0.645f, 0.051f, 0.534f}, {3.79f, 0.f, 0.237f, 0.446f, 2.77f, 0.523f, 0.042f, 0.467f}}},
      {422, 64, 128, 2, {{3.12f, 0.101f, 0.376f, 0.282f, 3.72f, 0.47f, 0.035f, 0.382f}, {4.15f, 0.511f, 0.591f, 0.264f, 3.55f, 0.447f, 0.018f, 0.322f}}},
      {610, 96, 64, 2, {{2.88f, 0.042f, 0.154f, 0.473f, 2.29f, 0.652f, 0.042f, 0.553f}, {4.46f, 0.f, 0.323f, 0.481f, 2.67f, 0.524f, 0.031f, 0.513f}}},
      {620, 96, 128, 2, {{3.67f, 0.442f, 0.513f, 0.251f, 3.35f, 0.511f, 0.025f, 0.413f}, {3.21f, 2.03f, 0.678f, 0.261f, 3.37f, 0.491f, 0.019f, 0.439f}}},
      {640, 96, 256, 3, {{2.63f, 3.97f, 1.22f, 0.f, 3.06f, 0.409f, 0.012f, 0.298f}, {2.59f, 4.58f, 1.55f, 0.f, 3.65f, 0.371f, 0.008f, 0.27f}}},
      {820, 128, 128, 3, {{2.16f, 2.88f, 0.848f, 0.f, 2.99f, 0.541f, 0.015f, 0.491f}, {2.19f, 3.49f, 1.08f, 0.f, 3.37f, 0.49f, 0.016f, 0.456f}}},
      {1020, 160, 128, 3, {{1.6f, 3.67f, 1.f, 0.f, 3.23f, 0.499f, 0.021f, 0.47f}, {2.15f, 3.61f, 1.39f, 0.f, 3.92f, 0.43f, 0.016f, 0.412f}}},
      {1620, 256, 128, 2, {{2.5f, 3.31f, 0.f, 1.64f, 3.07f, 0.497f, 0.013f, 0.481f}, {3.12f, 4.23f, 2.03f, 0.f, 3.22f, 0.436f, 0.004f, 0.427f}}}};
  // columns of the form's tiles; a width that N is no multiple of: launch_gemm() goes on to the kernels of gemm_decode.h
  const int width = code >= 5000 ? code / 10 % 10 * 32 : code == 1024 || code == 1025 || code == 512 ? 256 : code == 2560 ? 512 :
                    code == 2561 ? 320 : code == 256 || code == 768 || code == 769 || code == 1280 || code == 1281 ? 128 : 64;
  if (code < 0 || N % 64 != 0 || K % 64 != 0 || N % width != 0) return Q4Form{6, max(code, 0), sk};
  if (code == 0 && norm) return Q4Form{6, 0, 0};   // (the tile kernels there sum the squares of a row in an order of their own)
  const int nz = code == 0 ? 1 : prefill_slices(M, N, K, code, sk, slab_bytes);
  if ((code == 1025 || code == 769) && (sk == 0 || nz != sk)) return Q4Form{1, code, sk};   // (whole rounds, or partials only it has room for)
  static const int cus = [] {
    int v = 0, dev = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev);
    return v > 0 ? v : 256;
  }();
  const float weights = 1e-6f * (float)N * (float)K, omb = 2e-6f * (float)M * (float)N;
  const PrefillForm copy = prefill_form_cut(M, N, K, norm, rows16, slab_bytes, nz);
  Q4Form best = copy.us < 1e30f ? Q4Form{1, copy.code, nz} : Q4Form{code == 0 ? 6 : 1, code, sk};
  if (!group128 || !rows16 || K % 128 != 0) return best;
  const float part = copy.code == 1024 && nz > 2 ? 0.95f : copy.code >= 5000 && nz == 1 ? 0.82f : 0.87f;
  float least = part * (2.2f + 0.56f * weights + copy.us);
  auto over = [](int64_t x, int64_t y) { return (int)((x + y - 1) / y); };
  for (const Tile& t : tiles) {
    const int kts = over(K / 128, nz), full = 160 * 1024 / (t.stages * (t.bn * 64 + t.bm * 256 + 2048) + (norm ? q4_gamma_lds(K, nz) : 0));
    const int per_cu = t.code == 1620 ? 1 : full;   // (which fits whatever the slice)
    if (N % t.bn != 0 || per_cu == 0) continue;
    const int64_t blocks = (int64_t)over(M, t.bm) * (N / t.bn) * nz;
    const auto& x = t.cost[norm ? 1 : 0];
    const int rounds = over(blocks, (int64_t)cus * min(per_cu, 4));
    const float us = x.e + x.a * rounds + (x.b * over(blocks, cus) + x.g * rounds) * kts + x.w * 2.f * weights + x.o * omb +
                     (nz > 1 ? x.c + x.d * 2.f * nz * omb : 0.f);
    if (us < least) {
      least = us;
      best = Q4Form{5, t.code, nz};
    }
  }
  return best;
}

bool launch_q4_prompt(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.group != 128 || g.N % 64 != 0 || g.K % 128 != 0 || g.rownorm || g.ssp_in != nullptr || g.hg != nullptr ||
      g.ssp_out != nullptr || g.row_idx != nullptr || reinterpret_cast<uintptr_t>(g.x) % 16 != 0 || g.lda % 8 != 0 || g.lda >= (1 << 20) ||
      g.K >= (1 << 20) || g.scales == nullptr || g.zeros == nullptr ||
      ((reinterpret_cast<uintptr_t>(g.scales) | reinterpret_cast<uintptr_t>(g.zeros) | reinterpret_cast<uintptr_t>(g.norm_w)) & 15) != 0)
    return false;
  GemmParams p{};
  p.x = g.x; p.lda = g.lda; p.M = g.M;
  p.wp = reinterpret_cast<const uint4*>(g.wp); p.N = g.N; p.K = g.K;
  p.norm_w = g.norm_w; p.eps = g.eps;
  p.bias = g.bias; p.res = g.res; p.ldr = g.ldr;
  p.out = g.out; p.ldo = g.ldo;
  p.splitk = 1;
  p.slabs = g.slabs;
  p.positions = g.positions; p.slots = g.slots; p.cos_sin = g.cos_sin;
  p.k_cache = g.k_cache; p.v_cache = g.v_cache; p.hq = g.hq; p.hkv = g.hkv; p.bs = g.bs;
  p.scales = g.scales; p.zeros = g.zeros; p.group = g.group;
  p.dbg_ts = g.dbg_ts;
  int nz = g.splitk > 0 ? g.splitk : 1;
  while (nz > 1 && p.K / 64 / nz < 4) --nz;
  if (nz > 1 && (p.slabs == nullptr || ((size_t)nz * p.M * p.N + (size_t)nz * p.M) * 4 > g.slab_bytes)) nz = 1;
#define VG_Q4E(E) return g.norm_w != nullptr ? launch_q4_epi<E, true>(p, g.ntb, nz, st) : launch_q4_epi<E, false>(p, g.ntb, nz, st)
  switch (g.epi) {
    case EPI_SILU: VG_Q4E(EPI_SILU);
    case EPI_QKV: VG_Q4E(EPI_QKV);
    case EPI_F32: VG_Q4E(EPI_F32);
    default: VG_Q4E(EPI_BF16);
  }
#undef VG_Q4E
}

}  // namespace vgate
