// Operand copies padded to widths the 16-byte kernels take.  Widths that are
// not multiples of 8 put rows at 2- or 4-byte alignments; the general kernels
// handle them with element loads and per-tile conversions at a tenth of the
// fast kernels' rate.  One pass per operand makes op-dtype copies whose rows
// hold zeros up to the next multiple of 8 columns (zero products, zero
// contributions), 8 columns per thread.
#include "cvmm_common.h"
#include "cvmm_internal.h"

namespace cvmm {

// 8 columns from column c of a row of n, any alignment (the row's own
// element alignment): whole pieces as vector loads.
template <typename SrcT>
__device__ __forceinline__ void load8_row(const SrcT* __restrict__ row, int32_t c, int32_t n, float (&v)[8]) {
  if (c + 8 <= n) {
    SrcT e[8];
    __builtin_memcpy(e, row + c, sizeof(e));
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = to_f32(e[j]);
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = c + j < n ? to_f32(row[c + j]) : 0.f;
  }
}

// dst[r][0 .. n8) = rnd(src[r][c]) for c < n, 0 up to n8 = n rounded up to 8;
// with w: rnd(rnd(w[r]) * rnd(src[r][c])), the scaled rows of a weighted
// weight gradient.  Source row r is at (r / in_rows) * se + (r % in_rows) *
// ld where r % out_rows < in_rows, and zeros fill the other rows of each
// out_rows (an expert's matrix padded in both dimensions; plain rows have
// in_rows = out_rows = all of them).
template <typename SrcT, typename OpT>
__global__ __launch_bounds__(256) void pad_rows_kernel(const SrcT* __restrict__ src, int64_t se, int64_t ld,
                                                       int32_t n, int64_t chunks, FastDiv per_row, int32_t cpr,
                                                       FastDiv out_rows_div, int32_t in_rows, int32_t out_rows,
                                                       const void* __restrict__ w, int32_t w_dtype,
                                                       OpT* __restrict__ dst) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < chunks; i += (int64_t)gridDim.x * 256) {
    const int64_t r = per_row.div(i);
    const int32_t c = (int32_t)(i - r * cpr) * 8;
    const int64_t e = out_rows_div.div(r);
    const int32_t q = (int32_t)(r - e * out_rows);
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (q < in_rows) load8_row(src + e * se + q * ld, c, n, v);
    Chunk16 o;
    if (w != nullptr) {
      const float sc = round_to(load_as_f32(w, w_dtype, r), DTypeOf<OpT>::value);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        reinterpret_cast<OpT*>(&o)[j] = from_f32<OpT>(sc * to_f32(from_f32<OpT>(v[j])));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) reinterpret_cast<OpT*>(&o)[j] = from_f32<OpT>(v[j]);
    }
    *reinterpret_cast<uint4*>(dst + i * 8) = o.u;
  }
}

// `experts` blocks of in_rows source rows -> out_rows rows each.
static hipError_t launch_pad(const void* src, int32_t src_dtype, int64_t se, int64_t ld, int64_t n, int64_t experts,
                             int64_t in_rows, int64_t out_rows, const void* w, int32_t w_dtype, int32_t op_dtype,
                             void* dst, hipStream_t stream) {
  const int64_t cpr = (n + 7) / 8, chunks = experts * out_rows * cpr;
  if (chunks <= 0) return hipSuccess;
  if (chunks > 0x7fffffffll || out_rows > 0x7fffffffll || n > 0x7fffffffll) return hipErrorInvalidValue;
  int64_t blocks = (chunks + 255) / 256;
  if (blocks > 16384) blocks = 16384;
#define CVMM_PAD(S, O)                                                                                             \
  hipLaunchKernelGGL((pad_rows_kernel<S, O>), dim3((unsigned)blocks), dim3(256), 0, stream, (const S*)src, se, ld, \
                     (int32_t)n, chunks, make_fast_div(cpr), (int32_t)cpr, make_fast_div(out_rows), (int32_t)in_rows,       \
                     (int32_t)out_rows, w, w_dtype, (O*)dst)
  if (op_dtype == kBF16) {
    if (src_dtype == kF32) CVMM_PAD(float, bf16_t);
    else if (src_dtype == kBF16) CVMM_PAD(bf16_t, bf16_t);
    else return hipErrorInvalidValue;
  } else if (op_dtype == kF16) {
    if (src_dtype == kF32) CVMM_PAD(float, f16_t);
    else if (src_dtype == kF16) CVMM_PAD(f16_t, f16_t);
    else return hipErrorInvalidValue;
  } else {
    return hipErrorInvalidValue;
  }
#undef CVMM_PAD
  return hipGetLastError();
}

hipError_t launch_pad_rows(const void* src, int32_t src_dtype, int64_t ld, int64_t rows, int64_t n, const void* w,
                           int32_t w_dtype, int32_t op_dtype, void* dst, hipStream_t stream) {
  return launch_pad(src, src_dtype, 0, ld, n, 1, rows, rows, w, w_dtype, op_dtype, dst, stream);
}

// Expert matrices keys[e][i][j] with unit stride on `rows`' columns.
hipError_t launch_pad_matrices(const void* src, int32_t src_dtype, int64_t se, int64_t ld, int64_t experts,
                               int64_t rows, int64_t n, int32_t op_dtype, void* dst, hipStream_t stream) {
  return launch_pad(src, src_dtype, se, ld, n, experts, rows, pad8(rows), nullptr, 0, op_dtype, dst, stream);
}

// The transposed case of expert matrices: dst[e][j][i] = rnd(keys[e][i][j])
// padded in both dimensions, through a 64 x 64 LDS tile.
template <typename OpT>
__global__ __launch_bounds__(256) void pad_transpose_kernel(const void* __restrict__ keys, int32_t keys_dtype,
                                                            int64_t se, int64_t si, int64_t sj, int64_t d_i,
                                                            int64_t d_j, int64_t i8, int64_t j8,
                                                            OpT* __restrict__ dst) {
  __shared__ float tile[64][65];
  const int64_t e = blockIdx.z, i0 = (int64_t)blockIdx.y * 64, j0 = (int64_t)blockIdx.x * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int64_t i = i0 + r, j = j0 + tx;
    tile[r][tx] = i < d_i && j < d_j ? load_as_f32(keys, keys_dtype, e * se + i * si + j * sj) : 0.f;
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int64_t j = j0 + r, i = i0 + tx;
    if (i < i8 && j < j8) dst[(e * j8 + j) * i8 + i] = from_f32<OpT>(tile[tx][r]);
  }
}

hipError_t launch_pad_keys(const void* keys, int32_t keys_dtype, int64_t se, int64_t si, int64_t sj,
                           int32_t n_experts, int64_t d_i, int64_t d_j, int32_t op_dtype, void* dst,
                           bool transposed, hipStream_t stream) {
  const int64_t i8 = pad8(d_i), j8 = pad8(d_j);
  if (!transposed && sj == 1) return launch_pad_matrices(keys, keys_dtype, se, si, n_experts, d_i, d_j, op_dtype, dst, stream);
  if (transposed && si == 1) return launch_pad_matrices(keys, keys_dtype, se, sj, n_experts, d_j, d_i, op_dtype, dst, stream);
  // the transposed kernel writes [.][j][i]: swap the roles for [.][i][j]
  if (!transposed) return launch_pad_keys(keys, keys_dtype, se, sj, si, n_experts, d_j, d_i, op_dtype, dst, true, stream);
  if (n_experts > 65535 || (i8 + 63) / 64 > 65535) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((j8 + 63) / 64), (unsigned)((i8 + 63) / 64), (unsigned)n_experts);
  if (op_dtype == kBF16)
    hipLaunchKernelGGL(pad_transpose_kernel<bf16_t>, grid, dim3(256), 0, stream, keys, keys_dtype, se, si, sj, d_i,
                       d_j, i8, j8, (bf16_t*)dst);
  else if (op_dtype == kF16)
    hipLaunchKernelGGL(pad_transpose_kernel<f16_t>, grid, dim3(256), 0, stream, keys, keys_dtype, se, si, sj, d_i,
                       d_j, i8, j8, (f16_t*)dst);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace cvmm
