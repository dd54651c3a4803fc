// fp32 products on the matrix cores with DMA staging: the routed GEMM (forward
// and grad-input, cvmm.py:101-243, :363-421) and the per-expert weight
// gradient (cvmm.py:481-538) for fp32 operands whose rows are whole 16-byte
// pieces.
//
// What bounds them: the fp32 MFMA rate (64 flops per cycle and SIMD, 157
// TFLOP/s), 1/16 of the 16-bit one, so a 32-deep slice of a wave's 64 x 64
// block is 4096 cycles of MFMAs against a few hundred of LDS reads.  What matters is that every CU holds
// the same amount of work (small tiles), that a 64-row tile's shorter slices
// are requested two ahead (three buffers), and that nothing but MFMAs issues (the
// general kernel stages through registers, converting and transposing: a
// quarter of the rate).
//
// Column mapping: MFMA block i of a wave covers the columns NI c + i of its 16
// operand columns c (NI blocks), so one LDS read of NI consecutive columns
// feeds all NI blocks and a lane ends with NI consecutive columns of a row.
// Accumulation is fp32 throughout, in ascending slices of k (of routes).
#include "cvmm_gemm_panel.h"
#include "cvmm_wgrad_sched.h"

namespace cvmm {

typedef float f32xN4 __attribute__((ext_vector_type(4)));

template <int BM, int BN>
struct F32Cfg {
  static constexpr int STAGES = BM * BN > 64 * 128 ? 2 : 3;
  static constexpr int BK = 32;                       // k per slice
  static constexpr int WR = BM / 2, WC = BN / 2;      // rows, columns of a wave (2 x 2 waves)
  static constexpr int MJ = WR / 16, NI = WC / 16;    // MFMA blocks of a wave
  static constexpr int A_BYTES = BM * BK * 4, B_BYTES = BN * BK * 4;
  static constexpr int SLICE = A_BYTES + B_BYTES;
  static constexpr int D = SLICE / 4096;              // DMA instructions per wave per slice
  static constexpr int A_INSTS = A_BYTES / 1024;
  static constexpr int OCC = BM * BN > 64 * 64 ? 2 : 3;
  static_assert(NI == 2 || NI == 4, "2 or 4 columns per lane");
};

// 16 bytes as 4 floats / 8 bytes as 2, waited for by lgkm0_tied.
__device__ __forceinline__ float lane_f(const lds_u32x4& v, int i) {
  const uint32_t u = i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
  return __uint_as_float(u);
}

template <int N>
__device__ __forceinline__ void tie(lds_u32x4 (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}
template <int N>
__device__ __forceinline__ void tie(lds_u32x2 (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}
__device__ __forceinline__ void lgkm0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int BM, int BN, bool BNC, bool DG>
__global__ __launch_bounds__(kGemmThreads, (F32Cfg<BM, BN>::OCC)) void routed_gemm_f32_kernel(const GemmParams p) {
  using Cfg = F32Cfg<BM, BN>;
  constexpr int MJ = Cfg::MJ, NI = Cfg::NI, BK = Cfg::BK;
  __shared__ __attribute__((aligned(1024))) char ring[Cfg::STAGES * Cfg::SLICE];
  __shared__ RouteMeta<BM> meta;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t n_ntiles = (p.N + BN - 1) / BN;
  const bool tiled = gemm_schedule<BM>(p, n_ntiles, meta);
  const int64_t ntile = uniform_i32(meta.group);
  const int64_t n0 = ntile * BN;
  if (!tiled) {
    zero_unrouted_cols<BM>(p, meta, gridDim.x / n_ntiles, n0, n0 + BN, ntile);
    return;
  }
  const int32_t expert = uniform_i32(meta.expert);

  // ---- DMA sources: instruction j of wave w fills slice bytes
  // [(w * D + j) * 1024, +1024): A rows of 32 k (8 chunks of 16 bytes), then
  // B rows ([n][k] rows of 32 k, or BNC [k][n] rows of BN columns).  Chunk c
  // of A row r sits at c ^ (r & 7), of a [n][k] B row at c ^ ((r / NI) & 7).
  const char* zero = reinterpret_cast<const char*>(g_cvmm_zero_page);
  const char* src[Cfg::D];
  int kc[Cfg::D];
#pragma unroll
  for (int j = 0; j < Cfg::D; ++j) {
    const int gi = wave * Cfg::D + j;
    const int q = gi * 64 + lane;
    if (gi < Cfg::A_INSTS) {
      const int row = q >> 3, c = (q & 7) ^ (row & 7);
      const int64_t ar = meta.arow[row];
      kc[j] = c * 4;
      src[j] = ar >= 0 ? reinterpret_cast<const char*>(p.a) + (ar * p.a_ld + c * 4) * 4 : nullptr;
    } else {
      const int qb = q - Cfg::A_INSTS * 64;
      if constexpr (BNC) {
        const int krow = qb / (BN / 4), c = qb % (BN / 4);
        const int64_t n = n0 + c * 4;
        kc[j] = krow;
        src[j] = n < p.N ? reinterpret_cast<const char*>(p.b) + ((int64_t)expert * p.b_se + krow * p.b_sk + n) * 4 : nullptr;
      } else {
        const int row = qb >> 3, c = (qb & 7) ^ ((row / NI) & 7);
        const int64_t n = n0 + row;
        kc[j] = c * 4;
        src[j] = n < p.N ? reinterpret_cast<const char*>(p.b) + ((int64_t)expert * p.b_se + n * p.b_sn + c * 4) * 4 : nullptr;
      }
    }
  }
  const int64_t b_adv = BNC ? p.b_sk * 4 : 4;
  auto issue = [&](int64_t s, char* buf) {
    const int64_t k0 = s * BK;
#pragma unroll
    for (int j = 0; j < Cfg::D; ++j) {
      const int64_t adv = wave * Cfg::D + j < Cfg::A_INSTS ? 4 : b_adv;
      const char* sp = src[j] != nullptr && k0 + kc[j] < p.K ? src[j] + k0 * adv : zero;
      dma16(sp, buf + (wave * Cfg::D + j) * 1024);
    }
  };

  // ---- fragments: 16 k per step; lane (c = l % 16, q = l / 16) takes k =
  // 16 st + 4 q + e in MFMA e of the step, for both operands
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, fq = lane >> 4;
  f32x4_t acc[MJ][NI];
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const char* buf) {
    const uint32_t a_base = lds_addr(buf), b_base = a_base + Cfg::A_BYTES;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      lds_u32x4 af[MJ];
#pragma unroll
      for (int j = 0; j < MJ; ++j) {
        const int r = wm * Cfg::WR + j * 16 + fr;
        af[j] = lds_read128_at<0>(a_base + r * 128 + (((st * 4 + fq) ^ (r & 7)) << 4));
      }
      if constexpr (!BNC) {
        lds_u32x4 bf[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int r = wn * Cfg::WC + fr * NI + i;
          bf[i] = lds_read128_at<0>(b_base + r * 128 + (((st * 4 + fq) ^ ((r / NI) & 7)) << 4));
        }
        lgkm0();
        tie(af);
        tie(bf);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < MJ; ++j)
#pragma unroll
            for (int i = 0; i < NI; ++i)
              acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(lane_f(af[j], e), lane_f(bf[i], e), acc[j][i], 0, 0, 0);
      } else {
        using Vec = std::conditional_t<NI == 4, lds_u32x4, lds_u32x2>;
        Vec bf[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t at = b_base + (st * 16 + fq * 4 + e) * (BN * 4) + (wn * Cfg::WC + fr * NI) * 4;
          if constexpr (NI == 4) bf[e] = lds_read128_at<0>(at);
          else bf[e] = lds_read64(at);
        }
        lgkm0();
        tie(af);
        tie(bf);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < MJ; ++j)
#pragma unroll
            for (int i = 0; i < NI; ++i) {
              const uint32_t u = bf[e][i];
              acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(lane_f(af[j], e), __uint_as_float(u), acc[j][i], 0, 0, 0);
            }
      }
    }
  };

  const int64_t nk = (p.K + BK - 1) / BK;
  constexpr int STAGES = Cfg::STAGES;
#pragma unroll
  for (int s0 = 0; s0 < STAGES - 1; ++s0) {
    issue(s0, ring + s0 * Cfg::SLICE);  // (slices past K bring zeros)
    issue_fence();
  }
  int cur = 0;
  for (int64_t s = 0; s < nk; ++s) {
    vm_wait<(STAGES - 2) * Cfg::D>();  // slice s has landed (this wave's part; the other waves' after the barrier)
    wg_barrier();                      // ... and every wave is done with the buffer of slice s - 1
    issue(s + STAGES - 1, ring + (cur == 0 ? STAGES - 1 : cur - 1) * Cfg::SLICE);
    issue_fence();
    multiply(ring + cur * Cfg::SLICE);
    cur = cur + 1 == STAGES ? 0 : cur + 1;
  }
  vm_wait<0>();  // the zero slices past K, before the LDS is used again or released

  // ---- epilogue: lane holds rows wm*WR + 16 j + 4 fq + v, columns n0 + wn*WC + NI fr + [0, NI)
  const int64_t nl = n0 + wn * Cfg::WC + fr * NI;
  const bool n_in = nl < p.N;  // (N % 4 == 0: a lane's columns are all in or out)
  const bool has_w = p.w != nullptr;
  if (p.out != nullptr && n_in) {
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = wm * Cfg::WR + j * 16 + fq * 4 + v;
        const int64_t orow = meta.orow[m];
        if (orow < 0) continue;
        float x[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) x[i] = has_w ? acc[j][i][v] * meta.w[m] : acc[j][i][v];
        float* d = static_cast<float*>(p.out) + orow * p.out_ld + nl;
        if constexpr (NI == 4) *reinterpret_cast<float4*>(d) = make_float4(x[0], x[1], x[2], x[3]);
        else *reinterpret_cast<float2*>(d) = make_float2(x[0], x[1]);
      }
  }
  if constexpr (DG) {
    // routing-weight gradient partial of this n tile: sum_n acc[m][n] * x[m][n]
    // in a fixed order (a lane's columns, the 16 lanes of a row by xor 1, 2,
    // 4, 8, the two waves of the row)
    __syncthreads();
    float* red = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = wm * Cfg::WR + j * 16 + fq * 4 + v;
        const int64_t xr = meta.dgrow[m];
        float s = 0.f;
        if (xr >= 0 && n_in) {
          const float* x = static_cast<const float*>(p.dg_x) + xr * p.dg_x_ld + nl;
#pragma unroll
          for (int i = 0; i < NI; ++i) s += acc[j][i][v] * x[i];
        }
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) s += __shfl_xor(s, d, 64);
        if (fr == 0) red[wn * BM + m] = s;
      }
    __syncthreads();
    for (int m = tid; m < meta.rows; m += kGemmThreads)
      if (meta.widx[m] >= 0) p.dg[meta.widx[m] * p.dg_ntiles + ntile] = red[m] + red[BM + m];
  }
}

// Products from which a launch that the plain-FMA kernels (cvmm_small.hip)
// could run comes here instead: their latency is lower (three kernels of a
// 2048-route, 256 x 64 step 57 us against 64), their rate a third (2000
// routes of 512 x 128: 104 us against 73; 8000 of 256 x 64: 98 against 102).
// Launches those kernels cannot run (routing weights, the routing-weight
// gradient, wide outputs) come here at any size: a weighted 256-route, 64 x
// 256 step 57 us against the general kernels' 81, 16000 routes 130 against 323.
static bool f32_outweighs_small(int64_t n_routes, int64_t K, int64_t N) {
  return (double)n_routes * (double)K * (double)N >= 1.0e8;
}

bool f32_gemm_eligible(const GemmParams& p, int32_t op) {
  auto al = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const bool b_k = p.b_sk == 1 && p.b_sn % 4 == 0, b_n = p.b_sn == 1 && p.b_sk % 4 == 0;
  if (!(op == kF32 && p.a_dtype == kF32 && p.b_dtype == kF32 && p.K % 4 == 0 && p.N % 4 == 0 && p.n_out == p.N &&
        p.a_ld % 4 == 0 && p.b_se % 4 == 0 && al(p.a) && al(p.b) && (b_k || b_n) && p.epi == kEpiStore && p.act == 0 &&
        p.val_dtype == kF32 && (p.w == nullptr || p.prod_dtype < 0 || p.prod_dtype == kF32)))
    return false;
  if (p.out != nullptr && !(p.out_dtype == kF32 && p.out_ld % 4 == 0 && al(p.out))) return false;
  if (p.out == nullptr && p.dg == nullptr) return false;
  if (p.dg != nullptr && !(p.dg_x_dtype == kF32 && p.dg_val_dtype == kF32 && p.dg_x_ld % 4 == 0 && al(p.dg_x) &&
                           p.dg_ntiles == (p.N <= 64 ? 1 : (p.N + 127) / 128)))
    return false;
  return !small_gemm_eligible(p, op) || f32_outweighs_small(p.n_routes, p.K, p.N);
}

template <int BM, int BN>
static hipError_t launch_f32_gemm_t(const GemmParams& p_in, hipStream_t stream) {
  GemmParams p = p_in;
  p.token_major = resolve_token_major(p);
  const int64_t m_tiles = (p.n_routes + BM - 1) / BM + (p.n_experts < p.n_routes ? p.n_experts : p.n_routes);
  const int64_t grid = m_tiles * ((p.N + BN - 1) / BN);
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffll) return hipErrorInvalidValue;
  const bool bnc = p.b_sk != 1;
#define CVMM_F32(BNC, DG)                                                                                   \
  hipLaunchKernelGGL((routed_gemm_f32_kernel<BM, BN, BNC, DG>), dim3((unsigned)grid), dim3(kGemmThreads), 0, \
                     stream, p)
  if (p.dg != nullptr) {
    if (bnc) CVMM_F32(true, true);
    else CVMM_F32(false, true);
  } else {
    if (bnc) CVMM_F32(true, false);
    else CVMM_F32(false, false);
  }
#undef CVMM_F32
  return hipGetLastError();
}

// Tile: the one with the least work on the fullest CU, counted in tile areas
// (tile count estimated as R / BM + E / 2, 256 CUs; smaller tiles charged for
// their extra operand traffic, by what they take where every CU has many: 64
// experts, 32768 routes, 128 -> 1024 114 / 122 / 130 us with 128 x 128, 64 x
// 128 and 64 x 64).  1024 -> 128 143 / 125 / 113, 12 experts, 4000 routes, 1024
// -> 512 85 / 84 / 71, 4 experts, 700 routes, 1024 -> 1024 83 / 51 / 36: the
// rule's tile is the fastest of the three in each.  With the routing-weight
// gradient the columns stay at its partials' width.
hipError_t launch_f32_gemm(const GemmParams& p, hipStream_t stream) {
  auto cost = [&](int64_t bm, int64_t bn, double charge) {
    const int64_t tiles = ((p.n_routes + bm - 1) / bm + p.n_experts / 2) * ((p.N + bn - 1) / bn);
    return (double)((tiles + 255) / 256) * (double)(bm * bn) * charge;
  };
  const bool narrow = p.N <= 64;
  const bool fix_n = p.dg != nullptr || narrow;
  const double c128 = cost(128, narrow ? 64 : 128, 1.0), c64 = cost(64, narrow ? 64 : 128, 1.06);
  const double c64n = fix_n ? 1e300 : cost(64, 64, 1.15);
  if (narrow) return c128 <= c64 ? launch_f32_gemm_t<128, 64>(p, stream) : launch_f32_gemm_t<64, 64>(p, stream);
  if (c128 <= c64 && c128 <= c64n) return launch_f32_gemm_t<128, 128>(p, stream);
  if (c64 <= c64n) return launch_f32_gemm_t<64, 128>(p, stream);
  return launch_f32_gemm_t<64, 64>(p, stream);
}

// ---------------------------------------------------------------------------
// weight gradient: both operands are gathered route rows ([route][column] in
// LDS); lane (c, q) reads NJ consecutive x columns and NI consecutive dY
// columns of route 4 g + q: operands of MJ x NI MFMAs of 4 routes each.
// ---------------------------------------------------------------------------
template <int BM, int BN>
struct F32WgCfg {
  static constexpr int STAGES = BM * BN > 64 * 128 ? 2 : 3;
  static constexpr int BK = 32;  // routes per slice
  static constexpr int WR = BM / 2, WC = BN / 2, MJ = WR / 16, NI = WC / 16;
  static constexpr int A_BYTES = BM * BK * 4, B_BYTES = BN * BK * 4, SLICE = A_BYTES + B_BYTES;
  static constexpr int D = SLICE / 4096, A_INSTS = A_BYTES / 1024;
  static constexpr int OCC = BM * BN > 64 * 64 ? 2 : 3;
  static constexpr int TBL = 512;  // routes resolved at a time
};

template <int BM, int BN, bool WEIGHTED>
__global__ __launch_bounds__(kGemmThreads, (F32WgCfg<BM, BN>::OCC)) void wgrad_f32_kernel(const WgradParams p) {
  using Cfg = F32WgCfg<BM, BN>;
  constexpr int MJ = Cfg::MJ, NI = Cfg::NI, BK = Cfg::BK, TBL = Cfg::TBL;
  __shared__ __attribute__((aligned(1024))) char ring[Cfg::STAGES * Cfg::SLICE];
  __shared__ int32_t t_x[TBL], t_g[TBL];
  __shared__ float t_w[WEIGHTED ? TBL : 1];
  __shared__ WgSched sc;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t tiles_n = (p.N + BN - 1) / BN, tiles = ((p.M + BM - 1) / BM) * tiles_n;
  int64_t slot_id, tile;  // (grid = round_up(chunks, 8) * tiles)
  if (p.order == kWgOrderChunkXcd) {
    wgrad_chunk_xcd(blockIdx.x, (uint32_t)tiles, &slot_id, &tile);
  } else {
    slot_id = blockIdx.x / (uint32_t)tiles;
    tile = blockIdx.x - (uint32_t)slot_id * (uint32_t)tiles;
  }
  const int64_t m0 = (tile / tiles_n) * BM, n0 = (tile % tiles_n) * BN;
  if (!wgrad_schedule<kGemmThreads>(p, slot_id, sc, reinterpret_cast<int32_t*>(ring),
                                   kWgSortRoutes32))
    return;
  const int32_t expert = uniform_i32(sc.expert);
  const int64_t lo = sc.lo, hi = sc.hi;
  const int32_t nch = uniform_i32(sc.nch);

  // ---- DMA geometry: x rows of BM columns first, then dY rows of BN columns
  const char* zero = reinterpret_cast<const char*>(g_cvmm_zero_page);
  uint32_t tab[Cfg::D];
  const char* dbase[Cfg::D];
  int64_t dld[Cfg::D];
#pragma unroll
  for (int j = 0; j < Cfg::D; ++j) {
    const int gi = wave * Cfg::D + j;
    if (gi < Cfg::A_INSTS) {
      const int q = gi * 64 + lane, row = q / (BM / 4), c = (q % (BM / 4)) * 4;
      tab[j] = lds_addr(t_x + row);
      dbase[j] = m0 + c < p.M ? reinterpret_cast<const char*>(static_cast<const float*>(p.x) + m0 + c) : nullptr;
      dld[j] = p.x_ld * 4;
    } else {
      const int q = (gi - Cfg::A_INSTS) * 64 + lane, row = q / (BN / 4), c = (q % (BN / 4)) * 4;
      tab[j] = lds_addr(t_g + row);
      dbase[j] = n0 + c < p.N ? reinterpret_cast<const char*>(static_cast<const float*>(p.g) + n0 + c) : nullptr;
      dld[j] = p.g_ld * 4;
    }
  }
  auto issue = [&](int s, char* buf) {
    int32_t r[Cfg::D];
#pragma unroll
    for (int j = 0; j < Cfg::D; ++j) r[j] = lds_read_i32<0>(tab[j] + s * (BK * 4));
    lgkm_wait_tied(r);
#pragma unroll
    for (int j = 0; j < Cfg::D; ++j) {
      const char* src = r[j] >= 0 && dbase[j] != nullptr ? dbase[j] + (int64_t)r[j] * dld[j] : zero;
      dma16(src, buf + (wave * Cfg::D + j) * 1024);
    }
  };

  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 15, fq = lane >> 4;
  f32x4_t acc[MJ][NI];
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  using VecA = std::conditional_t<MJ == 4, lds_u32x4, lds_u32x2>;
  using VecB = std::conditional_t<NI == 4, lds_u32x4, lds_u32x2>;
  const uint32_t a_off = fq * (BM * 4) + (wm * Cfg::WR + fr * MJ) * 4;
  const uint32_t b_off = Cfg::A_BYTES + fq * (BN * 4) + (wn * Cfg::WC + fr * NI) * 4;
  const uint32_t w_off = lds_addr(t_w) + fq * 4;
  auto compute = [&](int s, const char* buf) {
    const uint32_t base = lds_addr(buf);
    constexpr int G = 4;  // groups of 4 routes read together
#pragma unroll
    for (int h = 0; h < BK / 4 / G; ++h) {
      VecA a[G];
      VecB b[G];
      int32_t w[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int gr = h * G + g;
        if constexpr (MJ == 4) a[g] = lds_read128_at<0>(base + a_off + gr * (4 * BM * 4));
        else a[g] = lds_read64(base + a_off + gr * (4 * BM * 4));
        if constexpr (NI == 4) b[g] = lds_read128_at<0>(base + b_off + gr * (4 * BN * 4));
        else b[g] = lds_read64(base + b_off + gr * (4 * BN * 4));
        if constexpr (WEIGHTED) w[g] = lds_read_i32<0>(w_off + s * (BK * 4) + gr * 16);
      }
      lgkm0();
      tie(a);
      tie(b);
      if constexpr (WEIGHTED) {
#pragma unroll
        for (int g = 0; g < G; ++g) asm volatile("" : "+v"(w[g]));
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float bv[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const uint32_t u = b[g][i];
          bv[i] = __uint_as_float(u);
          if constexpr (WEIGHTED) bv[i] *= __int_as_float(w[g]);
        }
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
          const uint32_t u = a[g][j];
#pragma unroll
          for (int i = 0; i < NI; ++i)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(u), bv[i], acc[j][i], 0, 0, 0);
        }
      }
    }
  };

  for (int64_t seg = lo; seg < hi; seg += TBL) {
    const int n_rt = (int)((hi - seg) < TBL ? (hi - seg) : TBL);
    const int n_st = (n_rt + BK - 1) / BK;
    if (seg != lo) __syncthreads();  // every wave is done with the previous table and buffers
    for (int r = tid; r < n_st * BK; r += kGemmThreads) {
      int32_t xr = -1, gr = -1;
      float w = 0.f;
      if (r < n_rt) {
        const int64_t q = seg + r;
        const int64_t xi = p.x_idx[q], graw = p.g_idx[q];
        const int64_t gi = graw >= 0 && graw < 0x7fffffffll ? p.g_fdiv.div(graw) : -1;
        if (xi >= 0 && xi < p.x_rows && gi >= 0 && gi < p.g_rows) {
          xr = (int32_t)xi;
          gr = (int32_t)gi;
          if constexpr (WEIGHTED) {
            const int64_t wi = p.w_idx[q];
            w = wi >= 0 && wi < p.n_routes ? load_as_f32(p.w, p.w_dtype, wi) : 0.f;
          }
        }
      }
      t_x[r] = xr;
      t_g[r] = gr;
      if constexpr (WEIGHTED) t_w[r] = w;
    }
    __syncthreads();
    constexpr int STAGES = Cfg::STAGES;
#pragma unroll
    for (int s0 = 0; s0 < STAGES - 1; ++s0) {
      if (s0 < n_st) issue(s0, ring + s0 * Cfg::SLICE);
      issue_fence();
    }
    int cur = 0;
    for (int s = 0; s < n_st; ++s) {
      vm_wait_slices<Cfg::D, STAGES - 2>(n_st - 1 - s < STAGES - 2 ? n_st - 1 - s : STAGES - 2);
      wg_barrier();
      if (s + STAGES - 1 < n_st) issue(s + STAGES - 1, ring + (cur == 0 ? STAGES - 1 : cur - 1) * Cfg::SLICE);
      issue_fence();
      compute(s, ring + cur * Cfg::SLICE);
      cur = cur + 1 == STAGES ? 0 : cur + 1;
    }
  }

  // ---- lane holds dW[m0 + wm*WR + MJ (4 fq + v) + j][n0 + wn*WC + NI fr + [0, NI)]
  const int64_t nl = n0 + wn * Cfg::WC + fr * NI;
  auto store = [&](auto&& value) {
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t m = m0 + wm * Cfg::WR + MJ * (fq * 4 + v) + j;
        if (m >= p.M || nl >= p.N) continue;
        float* d = static_cast<float*>(p.dw) + (int64_t)expert * p.dw_se + m * p.dw_sm + nl;
        float x[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) x[i] = value(j, i, v);
        __builtin_memcpy(d, x, NI * 4);
      }
  };
  if (nch == 1) {
    store([&](int j, int i, int v) { return acc[j][i][v]; });
    return;
  }
  // an expert of several chunks: fp32 partials, summed in chunk order by the
  // last to arrive (splitk_*, cvmm_common.h)
  const int64_t slot = sc.slot;
  if (slot >= p.max_slots) return;  // cannot happen: the workspace holds 2R/split + 1 slots
  constexpr int PER = MJ * NI * 4;  // values per lane
  const int64_t tile_elems = (int64_t)BM * BN;
  float* mine = p.partial + (slot * tiles + tile) * tile_elems + wave * (64 * PER) + lane;
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        __hip_atomic_store(mine + ((j * NI + i) * 4 + v) * 64, acc[j][i][v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  splitk_published();
  __syncthreads();
  if (tid == 0) sc.last = splitk_arrive(p.counters + (int64_t)expert * tiles + tile, nch);
  __syncthreads();
  if (!sc.last) return;
  splitk_acquired();
  const float* first = p.partial + (sc.base_slot * tiles + tile) * tile_elems + wave * (64 * PER) + lane;
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int32_t c = 0; c < nch; ++c) {
    const float* q = first + c * tiles * tile_elems;
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          acc[j][i][v] += __hip_atomic_load(q + ((j * NI + i) * 4 + v) * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  store([&](int j, int i, int v) { return acc[j][i][v]; });
}

bool f32_wgrad_eligible(const WgradParams& p, int32_t op) {
  auto al = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return op == kF32 && p.x_dtype == kF32 && p.g_dtype == kF32 && p.M % 4 == 0 && p.N % 4 == 0 && p.x_ld % 4 == 0 &&
         p.g_ld % 4 == 0 && al(p.x) && al(p.g) && p.dw_dtype == kF32 && p.dw_sn == 1 &&
         p.x_rows <= 0x7fffffffll && p.g_rows <= 0x7fffffffll &&
         (!small_wgrad_eligible(p, op) || f32_outweighs_small(p.n_routes, p.M, p.N));
}

template <int BM, int BN>
static hipError_t launch_f32_wgrad_t(const WgradParams& p, hipStream_t stream) {
  const int64_t tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  const int64_t grid = (p.grid_chunks + 7) / 8 * 8 * tiles;
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffll) return hipErrorInvalidValue;
  if (p.w != nullptr)
    hipLaunchKernelGGL((wgrad_f32_kernel<BM, BN, true>), dim3((unsigned)grid), dim3(kGemmThreads), 0, stream, p);
  else
    hipLaunchKernelGGL((wgrad_f32_kernel<BM, BN, false>), dim3((unsigned)grid), dim3(kGemmThreads), 0, stream, p);
  return hipGetLastError();
}

// dW tile: 128 x 128 where that still makes eight tiles per CU, else 64 x 128
// (128 x 64 for a narrow dW), so that experts of unequal loads fill the CUs
// evenly.  1024 x 128, 64 experts with loads up to 2.2x the mean, 32768
// routes: 102 us against 106 (64 x 64) and 138 (128 x 128).
void f32_wgrad_tile(int64_t M, int64_t N, int32_t n_experts, int* bm, int* bn) {
  const bool wide = ((M + 127) / 128) * ((N + 127) / 128) * n_experts >= 8 * 256;
  *bn = N <= 64 ? 64 : 128;
  *bm = M <= 64 ? 64 : (wide || N <= 64) ? 128 : 64;
}

// Workgroup order: a slot's tiles one after another over all XCDs, or from 64
// experts the slots dealt to the XCDs (the tiles of a slot share its rows in
// one L2).  Fewer slots leave XCDs idle or uneven when dealt: 1024 x 1024, 720
// routes, spread / dealt, evenly loaded and by Zipf's law: 2 experts 27 / 74
// and 33 / 89 us, 9: 34 / 48 and 33 / 62, 32: 45 / 46 and 49 / 68, 64: 86 / 84
// and 86 / 98; 1024 x 128, 16384 routes: 48 experts 58 / 57 and 67 / 68, 64:
// 56 / 54 and 71 / 71.
int32_t f32_wgrad_order(int32_t n_experts) { return n_experts >= 64 ? kWgOrderChunkXcd : kWgOrderChunk; }

hipError_t launch_f32_wgrad(const WgradParams& p, hipStream_t stream) {
  int bm, bn;
  f32_wgrad_tile(p.M, p.N, p.n_experts, &bm, &bn);
  if (bn == 64) return bm == 64 ? launch_f32_wgrad_t<64, 64>(p, stream) : launch_f32_wgrad_t<128, 64>(p, stream);
  return bm == 64 ? launch_f32_wgrad_t<64, 128>(p, stream) : launch_f32_wgrad_t<128, 128>(p, stream);
}

}  // namespace cvmm
