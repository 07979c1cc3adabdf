// fp32 outputs and the pair activations other than SiLU on the register-stationary decode GEMM (gemm_kx.h), without a norm in front.
#include "gemm_kx.h"

namespace vgate {

// (called by launch_dense_kx, which has looked at the shape)
bool launch_dense_kx_out(const GemmArgs& g, hipStream_t st) {
  if (g.rownorm || g.ssp_in != nullptr) return false;
  const GemmParams p = kx_params(g);
  if (g.act != 0) return g.epi == EPI_SILU && kx_launch<false, EPI_GLU, 0>(p, g, st);
  return kx_launch<false, EPI_F32, 0>(p, g, st);
}

}  // namespace vgate
