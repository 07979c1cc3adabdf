// EPI_GLU instantiation of the decode / small-M GEMM family (gemm_decode.h): bf16 weights without a norm in front.
#include "gemm_decode.h"

namespace vgate {
template void dispatch_epi<EPI_GLU, false>(GemmParams, const GemmArgs&, hipStream_t);
}  // namespace vgate
