// bf16 instantiations of the register-stationary decode GEMM (gemm_kx.h): the dense decode
// projections with the same grid forms as the int4 kernel (WIDE one block per CU owning whole tiles,
// GROUP 1-4 tiles per block + K slices), every weight fragment of a wave requested at once.
#include "gemm_kx.h"

namespace vgate {

// Half tiles (kx_half_kernel): up to 8 rows without a norm in front, where they come to one workgroup per CU at most. us, the
// tile blocks of gemm_decode.h -> half tiles, at 1 / 4 / 8 rows: 512 x 512 3.2 -> 2.3 / 3.6 -> 2.8 / 4.1 -> 2.8, 1024 x 4096 5.5 -> 4.4 /
// 6.0 -> 5.0 / 6.5 -> 5.5, 1536 x 1536 4.5 -> 3.4 / 4.8 -> 3.6 / 4.6 -> 3.8, 2048 x 6144 8.3 -> 6.5 / 8.5 -> 6.8 / 8.3 -> 7.5. Each block reads all of x: with a
// longer K up to 4 rows only (512 x 8192 6.5 -> 5.9 / 6.9, 6.9 / 7.5, 8.1, 1536 x 8960 9.1 -> 7.2 / 9.4 -> 8.3 / 9.2, 9.6). Two rounds of them lose what
// they gain from some 2 MB of weights on (3072 x 1536 4.8 -> 4.3 / 5.0 -> 4.5 / 4.8, 5.2, 3072 x 4096 6.7, 6.9 / 7.2, 7.6 / 7.5, 9.0).
bool launch_kx_half(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.M > (g.K <= 6144 ? 8 : 4) || g.N % 16 != 0 || g.N / 8 > kx_cus() || g.K % 128 != 0 || g.norm_w != nullptr ||
      g.ar_world > 0 || g.rownorm || g.row_idx != nullptr || (g.epi != EPI_BF16 && g.epi != EPI_F32) || g.act != 0 || g.ssp_in != nullptr ||
      (g.ssp_out != nullptr && !g.ss8))
    return false;
  GemmParams p = kx_params(g);
  // (k-quads of a wave: 2, and so 6 waves at K = 1536, were ahead of 1 and 3 by 2 to 5 %; more only where 16 waves need them)
  const int KQ = g.K / 128, kqw = std::max(std::min(2, KQ), (KQ + 15) / 16), nw = (KQ + kqw - 1) / kqw;
  if (kqw > 5) return false;
  const dim3 grid(g.N / 8), block(64 * nw);
  const size_t lds = (size_t)nw * 256;
  if (p.dbg_ts == nullptr) p.dbg_ts = tl_take("kx_half", (int)grid.x);
  auto kern = [&](auto epi) {
    constexpr int EPI = decltype(epi)::value;
    return kqw == 1 ? kx_half_kernel<1, EPI> : kqw == 2 ? kx_half_kernel<2, EPI> : kqw == 3 ? kx_half_kernel<3, EPI>
         : kqw == 4 ? kx_half_kernel<4, EPI> : kx_half_kernel<5, EPI>;
  };
  if (g.epi == EPI_F32) hipLaunchKernelGGL(kern(std::integral_constant<int, EPI_F32>{}), grid, block, lds, st, p);
  else hipLaunchKernelGGL(kern(std::integral_constant<int, EPI_BF16>{}), grid, block, lds, st, p);
  return true;
}

// Where the launcher prefers this kernel to the tile blocks of gemm_decode.h, which ask for a wave's k-range in groups and so twice or for k-steps
// that it hasn't. us, tile blocks -> here, at 1 / 8 / 16 rows:
//   K <= 1280, one k-quad per wave: 1024 x 1024 (above 8 rows) 4.8 -> 4.2, 3072 x 1024 4.6 -> 3.9 / 4.5 -> 4.2 / 5.4 -> 4.3, 6144 x 1024 5.8 -> 5.0
//     / 5.8 -> 5.0 / 7.6 -> 5.5, 14336 x 512 6.4 -> 5.4 / 6.9 -> 5.5 / 7.7 -> 5.7, 28672 x 1024 12.9 -> 12.5 / 13.9 -> 12.7 / 15.0 -> 13.2
//   whole tiles per CU, up to 5, K <= 1536: 6144 x 1536 6.3 -> 6.0 / 6.8 -> 6.2 / 8.0 -> 6.8, 12288 x 1536 8.8, 9.0 / 9.6 -> 9.3 / 12.0 -> 9.8; K <= 2048 from
//     8 rows on: 10240 x 2048 10.3 -> 10.0 / 11.3 -> 10.2 / 13.6 -> 10.8, 6144 x 1792 6.7, 7.2 / 7.9 -> 7.4 / 9.1 -> 8.1, 4096 x 1792 5.3, 5.6 / 5.6, 6.0 / 6.3, 6.9
//   fewer tiles than CUs: to K = 2048 for 4 rows at most (3072 x 1536 4.7 -> 4.5 / 4.8, 4.8 / 5.6, 5.5, 3584 x 1792 about even); above 8 rows
//     slices of 16 k-quads at most (1024 x 4096 8.3 -> 7.2, 512 x 8192 9.1 -> 7.4, 2048 x 4096 8.6 -> 7.7; of 18, 24: 1536 x 4608 9.4, 9.6, 2048 x 6144 9.2, 10.6)
//   but a norm's sums handed over that no wave can ask for ahead (K % 256, ss_pre_n4), for up to 4 rows of short K and a tile per CU: 1536 x 128 at 1 row
//     3.7, 4.0, at 8 4.5 -> 4.1, 2080 x 640 4.2, 4.7 / 5.1 -> 4.8 (1152 x 896 4.5, 4.6 / 5.0 -> 4.9)
bool dense_kx_fits(const GemmArgs& g) {
  if (g.M > 16 || g.N % 16 != 0 || g.K % 128 != 0 || g.epi == EPI_QKV) return false;
  const int tiles = g.N / 16, ncu = kx_cus(), KQ = g.K / 128, each = (tiles + ncu - 1) / ncu;
  if (g.ssp_in != nullptr && g.M <= 4 && g.K % 256 != 0 && g.K <= 640 && tiles <= ncu) return false;
  if (g.K <= 1280) return true;
  if (tiles >= ncu) return each <= 5 && (g.K <= 1536 || (g.K <= 2048 && each >= 2 && each <= 4 && g.M >= 8));
  if (2 * tiles > ncu) return g.K <= 2048 && g.M <= 4;
  const int S = std::min(ncu / tiles, KQ / 16);
  return g.M > 8 && S >= 2 && (KQ + S - 1) / S <= 16;
}

bool launch_dense_kx(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.M > 16 || g.N % 16 != 0 || g.K % 128 != 0 || g.norm_w != nullptr || g.ar_world > 0 ||
      g.row_idx != nullptr || (g.ssp_in != nullptr && g.rownorm))
    return false;
  if (g.epi == EPI_F32 || g.act != 0) return launch_dense_kx_out(g, st);
  const GemmParams p = kx_params(g);
  const int norm = g.rownorm ? 2 : g.ssp_in != nullptr ? 3 : 0;
#define VG_KX(E)                                               \
  return norm == 2 ? kx_launch<false, E, 2>(p, g, st)          \
       : norm == 3 ? kx_launch<false, E, 3>(p, g, st)          \
                   : kx_launch<false, E, 0>(p, g, st)
  switch (g.epi) {
    case EPI_SILU: VG_KX(EPI_SILU);
    case EPI_QKV: VG_KX(EPI_QKV);
    default: VG_KX(EPI_BF16);
  }
#undef VG_KX
}

}  // namespace vgate
