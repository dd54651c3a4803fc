// Long-K routed GEMM with bf16_t operands and outputs (cvmm_gemm_ring.h).
#include "cvmm_gemm_ring.h"

namespace cvmm {
template hipError_t launch_routed_gemm_ring_out<bf16_t, bf16_t>(const GemmParams& p, hipStream_t stream);
}  // namespace cvmm
