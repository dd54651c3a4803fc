// Routed GEMM for calls with few routes per expert (inference on a handful of
// tokens): y[q] = x[arow(q)] @ W_e with the expert weights read as they are
// stored -- [E][K][N] rows of N values, fp32 or the 16-bit op type -- each
// weight once per tile of 16 (32) rows.  An expert that draws many of the few
// routes has several such tiles, whose re-reads are bounded by the rule's
// average and stay below what a cast of every expert's weights reads: 32
// tokens, top-8, 128 experts of 2048 x 512 in fp32 93 us per call drawn
// evenly, 66 by Zipf's law, 35 all on one expert (cast: 244 / 230 / 189).
//
// What bounds it: the weights of the experts that have routes, streamed from
// HBM.  The 128-row tiles of the long-K kernel need a converted copy of every
// expert's weights first (whole-tensor read and write) and keep one DMA slice
// per workgroup in flight.  Here a wave loads 32 k x BN columns per step
// straight into registers (8 rows of 16 bytes per lane, one step ahead of the
// MFMAs), converts fp32 weights to the op type there (the rounding the
// copy would have applied), and turns the 8 k values of a column into the
// MFMA operand by register permutes; the routes' rows are the other operand,
// read from L2.  K is split over the workgroup's waves, whose partial tiles
// are added in wave order through LDS (deterministic).
//
// Column mapping: lane l holds columns NL (l % 16) .. + NL of the tile, and
// MFMA block i covers the columns NL c + i of its 16 operand columns c, so a
// lane ends with NL consecutive columns of its rows.
#pragma once

#include "cvmm_gemm_common.h"
#include "cvmm_mfma.h"

namespace cvmm {

// MB: 16-row blocks per tile; NW: waves per workgroup (K split NW ways); NT:
// the weights are read past the caches (non-temporal loads).
typedef unsigned int decode_u32x4 __attribute__((ext_vector_type(4)));

template <typename OpT, typename BT, int MB, int NW, bool NT_>
__global__ __launch_bounds__(NW * 64) void routed_decode_kernel(const GemmParams p) {
  constexpr int BM = 16 * MB, NT = NW * 64;
  constexpr int NL = 16 / (int)sizeof(BT);  // columns per lane
  constexpr int BN = 16 * NL;
  __shared__ __attribute__((aligned(16))) float part[NW][16][BN + 4];
  __shared__ RouteMeta<BM> meta;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, fq = lane >> 4;
  const int64_t n_ntiles = (p.N + BN - 1) / BN;
  const bool tiled = gemm_schedule_tile<BM>(p, n_ntiles, meta);
  const int64_t n0 = (int64_t)uniform_i32(meta.group) * BN;
  if (!tiled) {
    zero_unrouted_cols<BM, NT>(p, meta, gridDim.x / n_ntiles, n0, n0 + BN, -1);
    return;
  }
  const int32_t expert = uniform_i32(meta.expert);

  // this wave's run of 32-k steps
  const int steps = (int)((p.K + 31) / 32);
  const int per = (steps + NW - 1) / NW;
  const int s0 = wave * per, s1 = s0 + per < steps ? s0 + per : steps;

  const int64_t n = n0 + fr * NL;  // this lane's first column (N % 8 == 0: all in or out)
  const BT* bp = static_cast<const BT*>(p.b) + (int64_t)expert * p.b_se + n;
  const bool n_in = n < p.N;
  auto load_w = [&](int s, uint4 (&w)[8]) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int64_t k = (int64_t)s * 32 + fq * 8 + r;
      if constexpr (NT_) {
        decode_u32x4 t = {0, 0, 0, 0};
        if (n_in && k < p.K) t = __builtin_nontemporal_load(reinterpret_cast<const decode_u32x4*>(bp + k * p.b_sk));
        w[r] = make_uint4(t.x, t.y, t.z, t.w);
      } else {
        w[r] = n_in && k < p.K ? *reinterpret_cast<const uint4*>(bp + k * p.b_sk) : make_uint4(0, 0, 0, 0);
      }
    }
  };
  uint4 w0[8], w1[8];
  uint4 a0[MB], a1[MB];
  // the first weights are requested before the route rows are known
  if (s0 < s1) load_w(s0, w0);
  gemm_route_meta<BM, NT>(p, meta);
  const char* arow[MB];
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const int64_t ar = meta.arow[j * 16 + fr];
    arow[j] = ar >= 0 ? static_cast<const char*>(p.a) + ar * p.a_ld * 2 : nullptr;
  }
  auto load_a = [&](int s, uint4 (&a)[MB]) {
    const int64_t k = (int64_t)s * 32 + fq * 8;
#pragma unroll
    for (int j = 0; j < MB; ++j)
      a[j] = arow[j] != nullptr && k < p.K ? *reinterpret_cast<const uint4*>(arow[j] + k * 2) : make_uint4(0, 0, 0, 0);
  };

  f32x4_t acc[MB][NL];
#pragma unroll
  for (int j = 0; j < MB; ++j)
#pragma unroll
    for (int i = 0; i < NL; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const uint4 (&w)[8], const uint4 (&a)[MB]) {
    if constexpr (sizeof(BT) == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const uint32_t u = i == 0 ? w[r].x : i == 1 ? w[r].y : i == 2 ? w[r].z : w[r].w;
          v[r] = __uint_as_float(u);
        }
        const uint4 b = pack_chunk<OpT>(v);
#pragma unroll
        for (int j = 0; j < MB; ++j) MfmaOp<OpT>::step(acc[j][i], a[j], b);
      }
    } else {
#pragma unroll
      for (int h = 0; h < 4; ++h) {  // columns 2h, 2h + 1: dword h of every row
        uint32_t d[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) d[r] = h == 0 ? w[r].x : h == 1 ? w[r].y : h == 2 ? w[r].z : w[r].w;
        const uint4 lo = make_uint4(__builtin_amdgcn_perm(d[1], d[0], 0x05040100), __builtin_amdgcn_perm(d[3], d[2], 0x05040100),
                                    __builtin_amdgcn_perm(d[5], d[4], 0x05040100), __builtin_amdgcn_perm(d[7], d[6], 0x05040100));
        const uint4 hi = make_uint4(__builtin_amdgcn_perm(d[1], d[0], 0x07060302), __builtin_amdgcn_perm(d[3], d[2], 0x07060302),
                                    __builtin_amdgcn_perm(d[5], d[4], 0x07060302), __builtin_amdgcn_perm(d[7], d[6], 0x07060302));
#pragma unroll
        for (int j = 0; j < MB; ++j) {
          MfmaOp<OpT>::step(acc[j][2 * h], a[j], lo);
          MfmaOp<OpT>::step(acc[j][2 * h + 1], a[j], hi);
        }
      }
    }
  };

  // two register sets, the next step's loads ahead of this step's MFMAs
  if (s0 < s1) {
    load_a(s0, a0);
    int s = s0;
    for (; s + 2 < s1; s += 2) {
      load_w(s + 1, w1);
      load_a(s + 1, a1);
      multiply(w0, a0);
      load_w(s + 2, w0);
      load_a(s + 2, a0);
      multiply(w1, a1);
    }
    if (s + 1 < s1) {
      load_w(s + 1, w1);
      load_a(s + 1, a1);
      multiply(w0, a0);
      multiply(w1, a1);
    } else {
      multiply(w0, a0);
    }
  }

  // ---- 16 rows at a time: the waves' partials through LDS, added in wave order
  constexpr int PIECES = 16 * (BN / 8);  // 8-column pieces of 16 rows
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    if (j * 16 >= meta.rows) break;
    if (j > 0) __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float* d = &part[wave][fq * 4 + v][fr * NL];
#pragma unroll
      for (int i = 0; i < NL; i += 4)
        *reinterpret_cast<float4*>(d + i) = make_float4(acc[j][i][v], acc[j][i + 1][v], acc[j][i + 2][v], acc[j][i + 3][v]);
    }
    __syncthreads();
    for (int pc = tid; pc < PIECES; pc += NT) {
      const int r = pc / (BN / 8), c = (pc % (BN / 8)) * 8;
      const int64_t orow = meta.orow[j * 16 + r];
      if (orow < 0 || n0 + c >= p.N) continue;
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const float4 lo = *reinterpret_cast<const float4*>(&part[w][r][c]);
        const float4 hi = *reinterpret_cast<const float4*>(&part[w][r][c + 4]);
        v[0] += lo.x; v[1] += lo.y; v[2] += lo.z; v[3] += lo.w;
        v[4] += hi.x; v[5] += hi.y; v[6] += hi.z; v[7] += hi.w;
      }
      const int64_t off = orow * p.out_ld + n0 + c;
      Chunk16 h;
#pragma unroll
      for (int q = 0; q < 8; ++q) reinterpret_cast<OpT*>(&h)[q] = from_f32<OpT>(v[q]);
      if (p.act != 0) {  // GELU of the product in the output type; the product to aux
        *reinterpret_cast<uint4*>(static_cast<OpT*>(p.aux) + off) = h.u;
#pragma unroll
        for (int q = 0; q < 8; ++q)
          reinterpret_cast<OpT*>(&h)[q] = from_f32<OpT>(gelu_erf(to_f32(reinterpret_cast<const OpT*>(&h)[q])));
      }
      *reinterpret_cast<uint4*>(static_cast<OpT*>(p.out) + off) = h.u;
    }
  }
}

// Sizes the kernel is taken for, by routes per expert (the average), against
// the other way: a cast of every expert's weights and the long- or small-K
// kernel for fp32 weights, the long-K kernel on the stored rows (or a copy,
// K <= 128) for 16-bit ones.  Measured per call, this kernel / the other way,
// 128 experts:
//   fp32  2048 x 512:  1 route 71 / 204 us, 8: 133 / 225, 20: 143 / 223, 32: 216 / 224
//   fp32  512 x 2048:  1: 82 / 205, 8: 127 / 229, 20: 136 / 230, 32: 271 / 227
//   bf16  512 x 2048:  1: 33 / 63, 8: 46 / 87, 16: 54 / 89, 32: 101 / 90
//   bf16 1024 x 1024:  1: 30 / 41, 8: 46 / 50, 16: 48 / 50, 20: 58 / 51
//   bf16  2048 x 512:  1: 33 / 40, 8: 60 / 66, 12: 48 / 45, 20: 63 / 47
inline bool decode_sizes_ok(int64_t n_routes, int32_t n_experts, int64_t K, int64_t N, int32_t b_dtype) {
  const int64_t per = b_dtype == kF32 ? 20 : K <= 1024 ? 16 : 8;
  return n_routes > 0 && n_routes <= per * n_experts && K % 8 == 0 && N % 8 == 0;
}

// Weights as stored (rows of N values, fp32 or the op type), 16-byte aligned
// rows everywhere, the product stored once in the op type.
inline bool decode_eligible(const GemmParams& p, int32_t op) {
  auto al = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const int64_t bv = p.b_dtype == kF32 ? 4 : 8;
  return (op == kBF16 || op == kF16) && p.role == 0 && decode_sizes_ok(p.n_routes, p.n_experts, p.K, p.N, p.b_dtype) &&
         p.a_dtype == op && (p.b_dtype == op || p.b_dtype == kF32) && p.out_dtype == op && p.val_dtype == op &&
         p.b_sn == 1 && p.b_sk % bv == 0 && p.b_se % bv == 0 && p.a_ld % 8 == 0 && p.out_ld % 8 == 0 && al(p.a) &&
         al(p.b) && al(p.out) && p.n_out == p.N && p.epi == kEpiStore && p.out != nullptr && p.w == nullptr && p.dg == nullptr &&
         p.xs_out == nullptr && (p.act == 0 || (p.aux != nullptr && al(p.aux)));
}

// Weights from which they are read past the caches: a tensor that fills half
// the 256 MB Infinity Cache is gone from it by its next use (the block's other
// projection lies between).  268 MB of bf16 weights, 32 tokens: 53 -> 48 us;
// 33 MB of fp32 ones, which repeated calls do find there: 10.0 -> 11.7 us.
constexpr int64_t kDecodeStreamBytes = int64_t(128) << 20;

template <typename OpT, typename BT, int MB, int NW>
hipError_t launch_routed_decode_t(const GemmParams& p, hipStream_t stream) {
  constexpr int BM = 16 * MB, BN = 16 * (16 / (int)sizeof(BT));
  const int64_t m_tiles = (p.n_routes + BM - 1) / BM + (p.n_experts < p.n_routes ? p.n_experts : p.n_routes);
  const int64_t grid = m_tiles * ((p.N + BN - 1) / BN);
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffll) return hipErrorInvalidValue;
  if (p.n_experts * p.K * p.N * (int64_t)sizeof(BT) >= kDecodeStreamBytes)
    hipLaunchKernelGGL((routed_decode_kernel<OpT, BT, MB, NW, true>), dim3((unsigned)grid), dim3(NW * 64), 0, stream, p);
  else
    hipLaunchKernelGGL((routed_decode_kernel<OpT, BT, MB, NW, false>), dim3((unsigned)grid), dim3(NW * 64), 0, stream, p);
  return hipGetLastError();
}

template <typename OpT, typename BT>
hipError_t launch_routed_decode_b(const GemmParams& p_in, hipStream_t stream) {
  GemmParams p = p_in;
  p.token_major = 0;
  constexpr int BN = 16 * (16 / (int)sizeof(BT));
  const int64_t experts = p.n_experts < p.n_routes ? p.n_experts : p.n_routes;
  const int64_t tiles = experts * ((p.N + BN - 1) / BN), steps = (p.K + 31) / 32;
  if (p.n_routes > 8 * p.n_experts) return launch_routed_decode_t<OpT, BT, 2, 4>(p, stream);
  // up to one tile per CU: more waves per tile, each a shorter run of k
  // (16-bit weights: 8 columns per lane, whose 16-wave form would spill).
  // Launch time with 4 / 8 / 16 waves, fp32: 64 tiles of 32 steps 15.5 / 12.3
  // / 10.6 us, 128 of 32 21 / 15.5 / 12.9, 64 of 16 12.1 / 9.5 / 8.7, 128 of 8
  // 9.4 / 7.8 / 8.3; 512 of 16 16.1 / 15.8 / 20.0, 4096 of 16 62 / 69 / 99.
  // 16-bit with 4 / 8: 64 of 32 12.0 / 10.0, 64 of 8 8.4 / 8.0, 256 of 4 8.1 /
  // 8.6, 2048 of 16 36 / 47.
  if constexpr (sizeof(BT) == 4) {
    if (tiles <= 256 && steps >= 16) return launch_routed_decode_t<OpT, BT, 1, 16>(p, stream);
  }
  if (tiles <= 256 && steps >= 8) return launch_routed_decode_t<OpT, BT, 1, 8>(p, stream);
  return launch_routed_decode_t<OpT, BT, 1, 4>(p, stream);
}

template <typename OpT>
hipError_t launch_routed_decode_op(const GemmParams& p, hipStream_t stream) {
  if (p.b_dtype == kF32) return launch_routed_decode_b<OpT, float>(p, stream);
  return launch_routed_decode_b<OpT, OpT>(p, stream);
}

}  // namespace cvmm
