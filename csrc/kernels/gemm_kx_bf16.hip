// bf16 instantiations of the register-stationary decode GEMM (gemm_kx.h): the dense decode
// projections with the same grid forms as the int4 kernel (WIDE one block per CU owning whole tiles,
// GROUP 1-4 tiles per block + K slices), every weight fragment of a wave requested at once.
#include "gemm_kx.h"

namespace vgate {

// Half tiles (kx_half_kernel): up to 8 rows, bf16 outputs without a norm in front, where they come to one workgroup per CU at most. us, the
// tile blocks of gemm_decode.h -> half tiles, at 1 / 4 / 8 rows: 512 x 512 3.2 -> 2.3 / 3.6 -> 2.8 / 4.1 -> 2.8, 1024 x 4096 5.5 -> 4.4 /
// 6.0 -> 5.0 / 6.5 -> 5.5, 1536 x 1536 4.5 -> 3.4 / 4.8 -> 3.6 / 4.6 -> 3.8, 2048 x 6144 8.3 -> 6.5 / 8.5 -> 6.8 / 8.3 -> 7.5. Each block reads all of x: with a
// longer K up to 4 rows only (512 x 8192 6.5 -> 5.9 / 6.9, 6.9 / 7.5, 8.1, 1536 x 8960 9.1 -> 7.2 / 9.4 -> 8.3 / 9.2, 9.6). Two rounds of them lose what
// they gain from some 2 MB of weights on (3072 x 1536 4.8 -> 4.3 / 5.0 -> 4.5 / 4.8, 5.2, 3072 x 4096 6.7, 6.9 / 7.2, 7.6 / 7.5, 9.0).
bool launch_kx_half(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.M > (g.K <= 6144 ? 8 : 4) || g.N % 16 != 0 || g.N / 8 > kx_cus() || g.K % 128 != 0 || g.norm_w != nullptr ||
      g.ar_world > 0 || g.rownorm || g.row_idx != nullptr || g.epi != EPI_BF16 || g.act != 0 || g.ssp_in != nullptr ||
      (g.ssp_out != nullptr && !g.ss8))
    return false;
  GemmParams p = kx_params(g);
  // (k-quads of a wave: 2, and so 6 waves at K = 1536, were ahead of 1 and 3 by 2 to 5 %; more only where 16 waves need them)
  const int KQ = g.K / 128, kqw = std::max(std::min(2, KQ), (KQ + 15) / 16), nw = (KQ + kqw - 1) / kqw;
  if (kqw > 5) return false;
  const dim3 grid(g.N / 8), block(64 * nw);
  const size_t lds = (size_t)nw * 256;
  if (p.dbg_ts == nullptr) p.dbg_ts = tl_take("kx_half", (int)grid.x);
  switch (kqw) {
    case 1: hipLaunchKernelGGL(kx_half_kernel<1>, grid, block, lds, st, p); return true;
    case 2: hipLaunchKernelGGL(kx_half_kernel<2>, grid, block, lds, st, p); return true;
    case 3: hipLaunchKernelGGL(kx_half_kernel<3>, grid, block, lds, st, p); return true;
    case 4: hipLaunchKernelGGL(kx_half_kernel<4>, grid, block, lds, st, p); return true;
    default: hipLaunchKernelGGL(kx_half_kernel<5>, grid, block, lds, st, p); return true;
  }
}

bool launch_dense_kx(const GemmArgs& g, hipStream_t st) {
  if (g.M <= 0 || g.M > 16 || g.N % 16 != 0 || g.K % 128 != 0 || g.norm_w != nullptr || g.ar_world > 0 ||
      g.row_idx != nullptr || g.epi == EPI_F32 || g.act != 0 || (g.ssp_in != nullptr && g.rownorm))
    return false;
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
