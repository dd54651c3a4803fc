// Few-routes-per-expert routed GEMM instantiations (see cvmm_gemm_decode.h).
#include "cvmm_gemm_decode.h"

namespace cvmm {

bool routed_gemm_decode_applies(const GemmParams& p, int32_t op) { return decode_eligible(p, op); }

bool routed_gemm_decode_sizes(int64_t n_routes, int32_t n_experts, int64_t K, int64_t N, int32_t b_dtype) {
  return decode_sizes_ok(n_routes, n_experts, K, N, b_dtype);
}

hipError_t launch_routed_gemm_decode(const GemmParams& p, int32_t op, hipStream_t stream) {
  return op == kBF16 ? launch_routed_decode_op<bf16_t>(p, stream) : launch_routed_decode_op<f16_t>(p, stream);
}

}  // namespace cvmm
