// Work schedule of the per-expert weight gradients: (expert, route chunk)
// slots, largest first.
#pragma once

#include "cvmm_common.h"
#include "cvmm_internal.h"

namespace cvmm {

struct WgSched {
  int32_t expert, nch, last;
  int64_t lo, hi, slot, base_slot;
};

// Experts the sorted order is computed for (one per thread), and the mean
// routes per expert from which it is: 16-bit kernels, fp32 ones, none.
constexpr int32_t kWgSortExperts = 256;
constexpr int64_t kWgSortRoutes16 = 768, kWgSortRoutes32 = 384, kWgNoSort = int64_t(1) << 40;
constexpr int kWgSchedScratch = 2 * kWgSortExperts + 4;
static_assert(kWgSortExperts == 4 * 64, "four flags");

// (expert, route chunk) of work slot `slot_id`.  An expert of n routes is cut
// into ceil(n / p.split) chunks of equal length (multiples of 32 routes; at
// least one chunk per expert).  Slots run over the experts by chunk length,
// longest first (ties by id), so that the long chunks start first and the
// short ones fill the end of the launch: a router's loads differ by 2x and
// more between experts, and in id order the launch ended on whichever expert
// came last (64 experts of 1024 x 128, 1024 routes each, loads up to 1.4 times
// that: 42 us per launch in id order, 40 sorted).  Id order stays
//  - for more than kWgSortExperts experts, and up to 8 (they are dealt to one
//    XCD each: 8 of 1024 x 4096, loads up to 1.4 times the mean, 182 us
//    sorted, 172 not);
//  - below `sort_routes` routes per expert, where ranking costs every
//    workgroup what it evens out: 512 of them on each of 16, 2048 x 512, 44.3
//    us sorted, 42.6 not; 18 on each of 122 experts 38 and 29;
//  - where no expert has more than 1.25 times the mean (1024 routes on each of
//    64, 1024 x 128: 38.2 us sorted; 34.5 by this test, as without it).
// Every workgroup computes the same order.  `scratch` is kWgSchedScratch ints
// of LDS, 16-byte aligned, free again when this returns.  Returns false
// (uniformly) past the last slot.
template <int NT>
__device__ __forceinline__ bool wgrad_schedule(const WgradParams& p, int64_t slot_id, WgSched& s, int32_t* scratch,
                                               int64_t sort_routes) {
  static_assert(NT >= kWgSortExperts, "one thread per sorted expert");
  const int tid = threadIdx.x, lane = tid & 63;
  auto range = [&](int32_t e, int64_t& st, int64_t& n) {
    st = n = 0;
    if (e < p.n_experts) {
      int64_t end = p.offsets[e], start = e > 0 ? p.offsets[e - 1] : 0;
      end = end < 0 ? 0 : (end > p.n_routes ? p.n_routes : end);
      start = start < 0 ? 0 : (start > p.n_routes ? p.n_routes : start);
      st = start;
      n = end > start ? end - start : 0;
    }
  };
  // (most launches split no expert: no division there)
  auto chunks_of = [&](int32_t e, int64_t n) -> int32_t {
    if (e >= p.n_experts) return 0;
    return n <= p.split ? 1 : (int32_t)((n + p.split - 1) / p.split);
  };
  auto chunk_len = [](int64_t n, int32_t nch) -> int64_t { return nch == 1 ? n : (n + nch - 1) / nch; };
  bool sorted = p.n_experts <= kWgSortExperts && p.n_experts > 8 && p.n_routes >= sort_routes * p.n_experts;
  int32_t* len = scratch;                    // chunk length of expert e
  int32_t* order = scratch + kWgSortExperts; // expert of rank r
  int32_t* flags = order + kWgSortExperts;   // whether a wave's experts are uneven
  // this thread's expert; wave 0's are the scan's first 64 in id order
  int64_t st0 = 0, n0 = 0;
  if (tid < 64 || sorted) range(tid, st0, n0);
  if (sorted) {
    if (tid < kWgSortExperts) {
      const int32_t nch = chunks_of(tid, n0);
      len[tid] = nch > 0 ? (int32_t)chunk_len(n0, nch) : -1;
      const bool uneven = __any(4 * n0 * p.n_experts > 5 * p.n_routes);
      if (lane == 0) flags[tid >> 6] = uneven;
    }
    __syncthreads();
    const int4 f = *reinterpret_cast<const int4*>(flags);
    sorted = (f.x | f.y | f.z | f.w) != 0;
    if (sorted && tid < p.n_experts) {
      const int32_t mine = len[tid];
      int32_t rank = 0;
      for (int32_t j = 0; j < p.n_experts; j += 16) {  // (entries past the last expert: -1)
        int4 o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = *reinterpret_cast<const int4*>(len + j + 4 * q);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int32_t at = j + 4 * q;
          rank += (o[q].x > mine || (o[q].x == mine && at < tid)) ? 1 : 0;
          rank += (o[q].y > mine || (o[q].y == mine && at + 1 < tid)) ? 1 : 0;
          rank += (o[q].z > mine || (o[q].z == mine && at + 2 < tid)) ? 1 : 0;
          rank += (o[q].w > mine || (o[q].w == mine && at + 3 < tid)) ? 1 : 0;
        }
      }
      order[rank] = tid;
    }
    if (sorted) __syncthreads();
  }
  if (tid < 64) {
    if (lane == 0) s.expert = -1;
    int32_t carry = 0, carry_multi = 0;
    for (int32_t base = 0; base < p.n_experts; base += 64) {
      const int32_t r = base + lane;
      const int32_t e = r < p.n_experts ? (sorted ? order[r] : r) : p.n_experts;
      int64_t st = st0, n = n0;
      if (sorted || base > 0) range(e, st, n);
      const int32_t nch = chunks_of(e, n);
      const int32_t multi = nch > 1 ? nch : 0;
      const int32_t incl = wave_incl_scan(nch) + carry, incl_m = wave_incl_scan(multi) + carry_multi;
      const int32_t excl = incl - nch;
      if (nch > 0 && slot_id >= excl && slot_id < incl) {
        const int64_t c = slot_id - excl;
        const int64_t step = (chunk_len(n, nch) + 31) / 32 * 32;
        const int64_t a = c * step < n ? c * step : n, b = (c + 1) * step < n && c + 1 < nch ? (c + 1) * step : n;
        s.expert = e;
        s.nch = nch;
        s.lo = st + a;
        s.hi = st + b;
        s.base_slot = incl_m - multi;
        s.slot = s.base_slot + c;
      }
      carry = __builtin_amdgcn_readlane(incl, 63);
      carry_multi = __builtin_amdgcn_readlane(incl_m, 63);
      if (slot_id < carry) break;
    }
  }
  __syncthreads();
  return s.expert >= 0;
}

// Chunk-per-XCD order: (slot, tile) of workgroup i where the tiles of one
// chunk run together on one XCD (i % 8) and ranks are dealt to the XCDs back
// and forth (0 .. 7, 7 .. 0), which evens their sums.
__device__ __forceinline__ void wgrad_chunk_xcd(uint32_t i, uint32_t tiles, int64_t* slot_id, int64_t* tile) {
  const uint32_t xcd = i % 8, local = i / 8, row = local / tiles;
  *slot_id = (int64_t)row * 8 + ((row & 1) ? 7 - xcd : xcd);
  *tile = local - row * tiles;
}

}  // namespace cvmm
