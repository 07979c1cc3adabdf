// Weight-streaming MFMA GEMMs for the decode / small-M regime on gfx950, with the
// transformer's neighbouring ops fused in so a decoder layer is 4 GEMM launches.
//
//   out[m][n] = epilogue( sum_k prologue(x)[m][k] * W[n][k] )
//
// Weights are pre-packed ONCE at load time into "fragment-major" order so that
// one wave-instruction of 16 B/lane reads 1 KiB of contiguous HBM that is
// exactly the A operand of v_mfma_f32_16x16x32_bf16:
//
//   Wp[nt][kt][lane][j] = W[16*nt + (lane & 15)][32*kt + 8*(lane >> 4) + j]
//
// No LDS staging of weights: in the M <= 64 regime each weight byte is used by one
// wave only, so the bytes go straight to VGPRs with non-temporal loads
// (cdna_hip_programming.md §5 'GEMV / M <= 16 decode weights').
//
// Decomposition: grid = (n-tile groups, m-chunks of 16*MB rows, SPLITK k-slices).
// Inside a block, W waves split the block's k-slice into contiguous ranges and
// their accumulators are reduced through LDS. With SPLITK > 1 every block writes
// an fp32 partial slab and the LAST-ARRIVING block of the tile (sc1 slab stores ->
// drain -> ticket atomic; sc1 slab loads: no L2-wide release/acquire fences, see
// common.h) sums the slabs and runs the epilogue — no second launch, and the
// small-N projections (o_proj / down_proj: 96 tiles) still fill all 256 CUs.
//
// Fusions:
//   NORM          : RMSNorm folded into the GEMM with a DEFERRED row scale:
//                   out = rsqrt(mean(x^2) + eps) * (bf16(x * w) @ W^T). The sum of squares
//                   is accumulated from the same x fragments the MFMA loop already loads
//                   (no prologue pass, no serial latency before the weight stream) and
//                   applied per row in the epilogue (RMSNorm never runs as a kernel);
//   row_idx       : rows gathered by index (LM head reads only sampled rows);
//   epilogues     : +bias, +residual (in place), SiLU(gate)*up,
//                   f32 logits, and QKV: bias + NeoX RoPE + paged KV-cache write
//                   (one 16-column tile holds 8 rotation pairs / 8 gate-up pairs; the
//                   partners sit on lanes l, l ^ 32, see gemm_epilogue.h).
//
// Orientation: D = Wfrag(A) x xfrag(B) -> lane holds D[n = 4(l>>4)+i][m = l&15]:
// 4 consecutive output columns of one row -> 8-byte stores.
//
// AWQ W4A16 variant: int4 weights in the same fragment order, 4 k-tiles per 16-B
// lane load ([nt][kt/4][lane][4] uint32, nibble j = element j), group-wise
// (scale, scale*zero) applied in registers before the bf16 MFMA.
// The kernel templates and their launch logic live in gemm_decode.h; each epilogue's
// instantiations are compiled in gemm_epi_{bf16,f32,silu,qkv}.hip.
#include <stdexcept>

#include "gemm_decode.h"

namespace vgate {

int g_dec_u = -100;  // -100: the launcher's rule; else the forced decode register group size (tests)
void set_dec_u(int u) { g_dec_u = u; }

VG_EXTERN_EPI(EPI_BF16)
VG_EXTERN_EPI(EPI_F32)
VG_EXTERN_EPI(EPI_SILU)
VG_EXTERN_EPI(EPI_QKV)
VG_EXTERN_EPI(EPI_BF16_AR)
extern template void dispatch_epi<EPI_GLU, false>(GemmParams, const GemmArgs&, hipStream_t);

// ---- AWQ prefill operand: int4 fragments -> bf16 fragments (same fragment order) ----
// Long AWQ steps run the LDS-tiled bf16 prefill kernel (gemm_prefill.hip) on a per-call scratch
// copy of ONE matrix, dequantised here in the packed layout the kernel reads: lane l's k-step
// fragment of tile nt is element-wise (v - z) * s [* gamma_k] of the int4 fragment that the decode
// kernels feed to the MFMA as raw8. Folding the RMSNorm gamma in here turns the gamma-in-registers
// prologue (which the prefill kernel does not take) into the row-scale-only mode. No bf16 copy of
// the model is kept: the scratch is the largest single matrix (gate_up: 55 MB for Qwen2.5-1.5B).
// One wave per (tile, k-quad), a lane 16 B of int4 in and 4 x 16 B of bf16 out. What bounds it is the bf16 copy's bytes; the wave's
// place comes from the grid and its group from one uniform division (1536 x 8960: 9.8 -> 8.7 us, 17920 x 1536: 15.7 -> 14.0, 28672 x
// 4096: 67 -> 55; with a 64-bit remainder and four divisions per thread before).
__global__ __launch_bounds__(256) void awq_dequant_packed_kernel(const uint4* __restrict__ wq,
                                                                 const bf16_t* __restrict__ scales,
                                                                 const bf16_t* __restrict__ sz,
                                                                 const bf16_t* __restrict__ gamma, uint4* __restrict__ out,
                                                                 int N, int K, int group) {
  const int KQ = K >> 7, lane = threadIdx.x & 63;
  const int nt = blockIdx.y, kq = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (kq >= KQ) return;
  const size_t tq = (size_t)nt * KQ + kq;
  const int n = nt * 16 + (lane & 15);
  const uint4 q = wq[tq * 64 + lane];
  const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
  float s[4], zs[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {  // (group is a multiple of 32: a k-step of 32 lies in one)
    const size_t at = (size_t)((kq * 4 + u) * 32 / group) * N + n;
    s[u] = bf2f(scales[at]);
    zs[u] = bf2f(sz[at]);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = (float)((qw[u] >> ((j & 1) * 16 + 4 * (j >> 1))) & 0xF) * s[u] - zs[u];
    if (gamma != nullptr) {
      float g8[8];
      unpack8(*reinterpret_cast<const uint4*>(gamma + (kq * 4 + u) * 32 + 8 * (lane >> 4)), g8);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] *= g8[j];
    }
    out[(tq * 4 + u) * 64 + lane] = pack8(f);
  }
}

void launch_awq_dequant(const void* wq, const uint16_t* scales, const uint16_t* sz, const uint16_t* gamma,
                        void* out, int N, int K, int group, hipStream_t st) {
  hipLaunchKernelGGL(awq_dequant_packed_kernel, dim3((K / 128 + 3) / 4, N / 16), dim3(256), 0, st,
                     reinterpret_cast<const uint4*>(wq), reinterpret_cast<const bf16_t*>(scales),
                     reinterpret_cast<const bf16_t*>(sz), reinterpret_cast<const bf16_t*>(gamma),
                     reinterpret_cast<uint4*>(out), N, K, group);
}

template <bool AWQ>
static void launch_dispatch(GemmParams p, const GemmArgs& g, hipStream_t st) {
  if constexpr (!AWQ) {
    if (g.act != 0) return dispatch_epi<EPI_GLU, false>(p, g, st);
  }
  switch (g.epi) {
    case EPI_SILU: dispatch_epi<EPI_SILU, AWQ>(p, g, st); break;
    case EPI_QKV: dispatch_epi<EPI_QKV, AWQ>(p, g, st); break;
    case EPI_F32: dispatch_epi<EPI_F32, AWQ>(p, g, st); break;
    default: dispatch_epi<EPI_BF16, AWQ>(p, g, st);
  }
}

static GemmParams to_params(const GemmArgs& g) {
  GemmParams p{};
  p.x = g.x; p.lda = g.lda; p.M = g.M; p.row_idx = g.row_idx;
  p.wp = reinterpret_cast<const uint4*>(g.wp); p.N = g.N; p.K = g.K;
  p.norm_w = g.norm_w; p.eps = g.eps;
  p.bias = g.bias; p.res = g.res; p.ldr = g.ldr;
  p.out = g.out; p.ldo = g.ldo;
  p.slabs = g.slabs; p.counters = g.counters;
  p.gran = nullptr; p.fault = g.fault;  // (granule split-K: set by the decode launchers when it fits)
  p.positions = g.positions; p.slots = g.slots; p.cos_sin = g.cos_sin;
  p.k_cache = g.k_cache; p.v_cache = g.v_cache; p.hq = g.hq; p.hkv = g.hkv; p.bs = g.bs;
  if (g.act != 0) set_glu(p, GluAct{g.act, g.limit, g.alpha});
  p.scales = g.scales; p.zeros = g.zeros; p.group = g.group; p.szp = g.awq_szp;
  p.dbg_ts = g.dbg_ts;
  p.hg = g.hg; p.hg_gamma = g.hg_gamma; p.ssp_out = g.ssp_out; p.ssp_in = g.ssp_in; p.ssn = g.ssn; p.ss8 = g.ss8;
  p.ar = ArFused{};
  if (g.ar_world > 0) {
    for (int r = 0; r < 8; ++r) p.ar.base[r] = g.ar_fused[r];
    p.ar.err = g.ar_err; p.ar.rank = g.ar_rank; p.ar.world = g.ar_world; p.ar.spin = ar_spin();
  }
  return p;
}

// What the medium kernel leaves of 17 .. 64 rows, long K of many columns and LM heads with a row gather, runs on the tiles of gemm_decode.h, which
// hold one stage of weights ahead and stage x anew for each block's k-range, or on four-wave tiles, three to five stages in flight: 64 x
// 64, two blocks to a CU, or 64 x 128. Whether: us, cold weights, tiles of gemm_decode.h -> four-wave tiles, at 17 / 64 rows.
//   With a norm folded in: 8320 x 2304 22.3 -> 14.2 / 26.3 -> 15.6, 16384 x 4096 51.7 -> 27.6 / 58.1 -> 29.0, 32000 x 1536 25.4 -> 21.9 / 29.4 -> 24.0,
//     151936 x 1536 96.2 -> 94.1 / 116 -> 114. But, not for pairs (131072 x 512 46 -> 40), K of one or two whole stages of the other kernels, 256 or 512, where their blocks of 128 columns fill
//     whole rounds of CUs: 65536 x 512, fp32, 20.3, 22.8 / 24.8, 27.6, 98304 x 512 28.0, 30.2 / 33.4, 36.2, 128256 x 256 22.4, 23.1 / 29.5, 28.7 (49152 x 512, three halves
//     of a round, 18.3 -> 16.6 / 21.2 -> 19.8, 151936 x 512 39.9 -> 38.8 / 49.1 -> 45.2; 65536 x 448 19.2 -> 17.3 / 23.5 -> 21.0, x 576 23.5 -> 20.0 / 28.3 -> 23.9).
//   Without one, up to 12288 columns from 25 rows on: 8320 x 4096 20.9, 21.2 / 28.9 -> 23.7. Wider, from K = 2048 on, by how well the other kernels fill the
//     chip. Pairs and QKV, 64 columns to a block of theirs, lose more of it with more rows: 17408 x 3072 32.1 -> 26.4 / 44.2 -> 30.9; up to 24 rows of
//     more than 28672 columns they are even or ahead (32000 x 6144 65.9, 72.6 / 87.9 -> 75.6). Others are 128 columns wide from 16384 on, one block to a
//     CU: with the last round of them four fifths full or less 16384 x 3072 29.4 -> 20.1 / 35.1 -> 22.1, 25600 x 3072 32.1 -> 31.8 / 37.9 -> 35.3, 40960 x
//     3072 59.3 -> 51.5 / 69.8 -> 58.4; fuller ones hold (32000 x 4096 48.7, 52.2 / 52.1, 54.4, 65536 x 2304 52.8, 58.7 / 65.7, 71.6, 128256 x 2304 104, 113 /
//     129, 141), but for more than 32 rows in a single round nine tenths full (27648 x 2304 25.9, 26.9 / 30.8 -> 28.5). Columns that are no multiple
//     of 128 run on the K-split kernels, which hold up to 24 rows (23360 x 3584 34.1, 37.4 / 60.7 -> 43.9).
static bool four_wave_fits(const GemmArgs& g) {
  if (g.norm_w != nullptr || g.N < 8192) return false;
  const int cus = cu_count_gemm();
  if (g.rownorm) {
    const int blocks = g.N / 128, slots = (blocks + cus - 1) / cus * cus;
    return g.epi == EPI_SILU || g.epi == EPI_QKV || g.N % 128 != 0 || g.K > 512 || g.K % 256 != 0 || blocks <= cus || 20 * blocks <= 19 * slots;
  }
  if (g.N <= 12288) return g.M > 24;
  if (g.K <= 2048) return false;
  if (g.epi == EPI_SILU || g.epi == EPI_QKV) return g.M > 24 || g.N <= 112 * cus;
  if (g.N % 128 != 0) return g.M > 24;
  const int blocks = g.N / 128, slots = (blocks + cus - 1) / cus * cus;
  return 10 * blocks <= 8 * slots || (g.M > 32 && 10 * blocks <= 9 * cus);
}
// 128 columns to a tile where the narrow ones come to more than one block per CU and these to one at most, and K is long enough for
// their six stages (64 x 64 / 64 x 128, us with a norm folded in, at 17 / 64 rows: 16384 x 4096 (128 blocks of 128) 27.6, 33.6 / 29.0, 39.4; 17408 x 4096
// 39.3 -> 34.8 / 46.4 -> 40.3; 24576 x 1024 13.9, 14.4 / 16.2, 16.2, x 1536 18.9 -> 18.7 / 22.1 -> 20.3, x 2304 26.4 -> 24.6 / 31.0 -> 27.0; 32000 x 1536 21.9,
// 22.6 / 24.7 -> 24.0, x 2048 27.3, 28.9 / 30.7 -> 30.4, x 2304 30.6, 30.6 / 34.6 -> 32.3; 33792 x 2304 (264 blocks) 39.0, 46.4 / 43.8, 49.9): K of 2048 at most
// and up to 32 rows want no more than three quarters of the CUs.
static bool four_wave_wide(const GemmArgs& g) {
  const int cus = cu_count_gemm(), blocks = g.N / 128;
  return g.N % 128 == 0 && 2 * blocks > cus && blocks <= cus && g.K >= 1536 && (g.K > 2048 || g.M > 32 || 4 * blocks <= 3 * cus);
}

void launch_gemm(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0) return;
  // TP row-parallel decode GEMM with the all-reduce in the epilogue: the tile-per-block decode kernels
  // (one wave finishes a whole 16-row tile: epilogue_ar's lane layout); the binding checked the shape
  if (g.ar_world > 0) {
    dispatch_epi<EPI_BF16_AR, false>(to_params(g), g, st);
    return;
  }
  // long steps (prefill chunks): the LDS-tiled MFMA kernel (gemm_prefill.hip) on the same packed
  // weights; it declines shapes / modes it does not take
  // mixed prefill + decode steps (16 < M <= 64): the medium-M kernel when the start-up tuner
  // measured it faster (path 2, gemm_mid.hip); it declines shapes / modes it does not take
  if (g.path == 2 && launch_gemm_mid(g, st)) return;
  if (g.path == 6) return launch_dispatch<false>(to_params(g), g, st);  // the kernels of gemm_decode.h (q4_prompt_form)
  // without a plan, 17 .. 64 rows: one block per CU owning whole tiles (wide) where K is short, K slices over narrow
  // tiles where it is long. us at 32 rows, the K-split / tile kernels of gemm_decode.h -> now: 17920 x 1536 18.3 -> 13.2, 6464 x 1536
  // 13.7 -> 7.2, 1536 x 8960 18.8 -> 12.8, 1024 x 4096 11.8 -> 7.9, 1536 x 1536 7.9 -> 5.1. Above 32 rows the wide form pays
  // once its tiles cover the CUs (N >= 4160; at 64 rows 6464 x 1536 17.5 -> 10.0; 1536 x 1536 8.1, sliced 7.5, at 48 5.9, 6.9). Long and wide stays
  // with the kernels below (8192 x 3072 at 64 rows 18.4, sliced 24.2), and so do up to 32 rows of 3072 to 4096 columns, which
  // fill the chip without slices (4096 x 4096 at 24 rows 11.4, sliced 13.3, at 32 13.1, 13.8, at 48 18.8 -> 14.8; with longer K sooner:
  // 3072 x 5120 at 32 16.4 -> 12.3), slices that come to little more than a workgroup per CU (2048 x 8960, 288 of them, at 17 rows 15.6, 15.8;
  // 6144 x 3072 at 17 14.5, 15.1) and the very shortest (1536 x 3072 at 17 rows 8.1, 8.5, at 24 9.1 -> 8.8).
  // A folded norm costs the wide form more than the K-split kernels, which have more waves to sum squares: few columns of K up to 1024 and of
  // 2048 stay with them (4096 x 1024 at 17 rows 5.3, wide 6.0, at 32 6.6, 6.4; 1024 x 2048 at 17 6.5, 6.6; 1024 x 1536 at 24 7.8 -> 6.1).
  // The lines were drawn before the medium kernel brought x by whole lines, which some it does not take would now be ahead with: 2048 x 8960 at 24
  // rows 17.3, sliced 15.9, at 64 27.0, 22.6; 3584 x 1792 at 48 12.0, wide 8.8; 1024 x 1024 at 48 6.6, wide 5.6; 1024 x 2048 with a norm at 32 8.5, 6.7.
  // (both stage rows of x by 16-B LDS-DMA: rows that are not 16-B aligned stay below)
  const bool rows16 = reinterpret_cast<uintptr_t>(g.x) % 16 == 0 && g.lda % 8 == 0;
  if (g.path == 0 && rows16 && g.M > 16 && g.M <= 64 && g.waves == 0 && g.splitk == 0 && g.ntb == 0 && g.N >= 512) {
    GemmArgs h = g;
    if (g.K > 2048) {
      const int64_t groups = g.N / 64;   // (workgroups per slice; slices of 32 k-steps at most, as launch_gemm_mid() cuts them)
      const int64_t blocks = groups * ((g.K + 1023) / 1024);
      const bool filled = g.N >= 3072 && g.N <= 4096 && g.M <= 32 && g.K <= (g.N > 3584 ? (g.M <= 24 ? 14336 : 5120) : 4096);
      const bool over = blocks > 256 && blocks <= 320 && (g.M <= 24 || g.N <= 4096);
      const bool shortest = g.M <= 20 && ((g.K <= 3072 && g.N <= 2048) || (g.rownorm && g.K <= 4096 && g.N > 4096 && g.N < 8192));
      h.waves = (g.N < 8192 || (g.N == 8192 && g.M <= 32)) && !filled && !over && !shortest ? 4 : 0;
    }
    else if (g.M <= 32) h.waves = g.rownorm && g.N <= 4096 && (g.K <= 1024 || g.K > 1792) ? 0 : 8;
    else if (g.N >= 4160) h.waves = 8;
    else if (g.K > 1024 && g.N <= 2048) h.waves = 4;
    if (h.waves != 0 && launch_gemm_mid(h, st)) return;
    if (four_wave_fits(g)) {
      h = g;
      h.ntb = four_wave_wide(g) ? 5240 : 5220;
      if (launch_gemm_prefill(h, st)) return;
    }
  }
  // decode rows without a plan: half tiles or the register-stationary kernel where those are ahead (gemm_kx_bf16.hip); path 4, a decode plan or
  // forced: the latter
  if (g.path == 0 && g.waves == 0 && g.splitk == 0 && g.ntb == 0 && (launch_kx_half(g, st) || (dense_kx_fits(g) && launch_dense_kx(g, st)))) return;
  if (g.path == 4) {
    GemmArgs h = g;
    if (h.ntb > -12 || h.ntb < -14) h.ntb = 0;
    if (launch_dense_kx(h, st)) return;
    h.path = 0; h.waves = 0; h.splitk = 0; h.ntb = 0;
    launch_dispatch<false>(to_params(h), h, st);
    return;
  }
  // decode rows on the stream-K kernel (path 3: a decode plan / forced), else the tile-per-block kernels
  if (g.path == 3) {
    if (launch_gemm_sk(g, st)) return;
    // declined (shape / mode / occupancy): a stream-K plan's (waves, blocks per CU, k-group) fields
    // mean nothing to the tile kernels — fall back on the launcher's own heuristic
    GemmArgs h = g;
    h.path = 0; h.waves = 0; h.splitk = 0; h.ntb = 0;
    launch_dispatch<false>(to_params(h), h, st);
    return;
  }
  // (65 .. 127 rows: the same forms unless K is short, where the kernels below are ahead: 512 x 512 at 80 rows 8.2, 9.2 us, 1024 x 512 8.4,
  // 9.0; from there on the forms: 1024 x 1024 at 96 rows 12.1 -> 10.6, 1536 x 1536 at 96 14.7 -> 12.3, 1536 x 8960 at 96 42 -> 19)
  const bool longer = g.M >= 128 || (g.M > 64 && rows16 && g.K >= 1024);
  if (g.path == 1 || (g.path == 0 && longer && g.waves == 0 && g.splitk == 0)) {
    GemmArgs h = g;
    if (g.path == 0) h.ntb = 0;
    if (launch_gemm_prefill(h, st)) return;
    if (h.ntb >= 5000) {  // rows off 16 B, a norm in registers or a row gather: the launcher's choice, a plan's numbers mean nothing below
      h.path = 0; h.ntb = 0; h.splitk = 0;
      return launch_gemm(h, st);
    }
  }
  launch_dispatch<false>(to_params(g), g, st);
}

void launch_awq_gemm(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0) return;
  if (g.ar_world > 0) {  // fused all-reduce: the K-split int4 kernel (gemm_finish -> epilogue_ar)
    GemmArgs h = g;
    h.ntb = -2;
    dispatch_epi<EPI_BF16_AR, true>(to_params(h), h, st);
    return;
  }
  // decode (M <= 16) on the register-stationary int4 kernel: the launcher's choice (no forced waves /
  // tiles per block), or g.ntb = -12 / -13 / -14 (1 / 2 / 4 tiles per block) with the forced waves / slices
  if (g.path == 0 && ((g.ntb == 0 && g.waves == 0) || (g.ntb <= -12 && g.ntb >= -14)) && launch_awq_kx(g, st)) return;
  // mixed prefill + decode steps (16 < M <= 64) on the int4 medium kernel (path 2)
  if (g.path == 2 && launch_awq_mid(g, st)) return;
  if (g.path == 5) {
    if (launch_q4_prompt(g, st)) return;
    throw std::runtime_error("gemm: the int4 prompt kernel does not take this tile, shape or alignment");
  }
  launch_dispatch<true>(to_params(g), g, st);
}

}  // namespace vgate