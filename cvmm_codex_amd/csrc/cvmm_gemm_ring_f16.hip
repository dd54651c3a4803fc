// Long-K routed GEMM with f16_t operands and outputs (cvmm_gemm_ring.h).
#include "cvmm_gemm_ring.h"

namespace cvmm {
template hipError_t launch_routed_gemm_ring_out<f16_t, f16_t>(const GemmParams& p, hipStream_t stream);
}  // namespace cvmm
