#include "gemm_prompt.h"

namespace vgate {

template <int MT, int NT, int NS, int EPI, int NORM>
static bool launch_w4_one(const GemmParams& p, int nz, hipStream_t st) {
  using G = W4<MT, NT>;
  if (p.N % G::BN != 0) return false;
  const int blocks = ((p.M + G::BM - 1) / G::BM) * (p.N / G::BN);
  GemmParams q = p;
  if (q.dbg_ts == nullptr) q.dbg_ts = tl_take("gemm_w4", blocks * nz);
  auto kern = gemm_w4_kernel<MT, NT, NS, EPI, NORM>;
  static bool attr = [&] {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, NS * G::STAGE) == hipSuccess;
  }();
  (void)attr;
  hipLaunchKernelGGL(kern, dim3(blocks, nz), dim3(256), NS * G::STAGE, st, q);
  return true;
}

// code: 5000 + 100 MT + 10 NT (gemm_prefill.hip lists them); false: not a tile of these, or not one of N
template <int EPI, int NORM>
bool launch_gemm_w4(const GemmParams& p, int code, int nz, hipStream_t st) {
  switch (code) {
#define VG_W4(MT, NT, NS) case 5000 + MT * 100 + NT * 10: return launch_w4_one<MT, NT, NS, EPI, NORM>(p, nz, st)
    VG_W4(2, 2, 4);  // two blocks to a CU
    VG_W4(2, 4, 6);
    VG_W4(3, 4, 5);
    VG_W4(3, 8, 3);
    VG_W4(5, 8, 3);
    VG_W4(6, 4, 4);
    VG_W4(6, 8, 2);  // (QKV with a norm spills 12 registers around its epilogue and is ahead all the same: 1792 rows, 6144 x 4096 122 us, 256 x 256 126)
#undef VG_W4
  }
  return false;
}
#define VG_W4_INST(E)                                                              \
  template bool launch_gemm_w4<E, 0>(const GemmParams&, int, int, hipStream_t);    \
  template bool launch_gemm_w4<E, 2>(const GemmParams&, int, int, hipStream_t);
VG_W4_INST(EPI_BF16)
VG_W4_INST(EPI_F32)
VG_W4_INST(EPI_SILU)
VG_W4_INST(EPI_QKV)
template bool launch_gemm_w4<EPI_GLU, 0>(const GemmParams&, int, int, hipStream_t);
#undef VG_W4_INST

}  // namespace vgate
