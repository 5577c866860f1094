// Rows of an append in tiles, and the INT4 group rescue's threshold over them (device code shared
// by append_bulk.hip and quant_append.hip).
#pragma once
#include "append_row.h"

#pragma clang fp contract(off)

namespace kvq {

namespace {

typedef int16_t i16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk_max_i(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(i16x2, a),
                                                                __builtin_bit_cast(i16x2, b)));
}
__device__ __forceinline__ uint32_t pk_min_i(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(i16x2, a),
                                                                __builtin_bit_cast(i16x2, b)));
}
template <int CTRL>
__device__ __forceinline__ uint32_t dppu(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, false);
}
// the value of the lane CTRL - 0x110 below in its row of 16, 0 past the row's start
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_shr(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, true);
}
__device__ __forceinline__ uint32_t swap16(uint32_t x) { return (x >> 16) | (x << 16); }

__device__ __forceinline__ uint32_t max_group(uint32_t m, int gs) {
  if (gs >= 16) m = pk_max_i(m, dppu<0xB1>(m));
  if (gs >= 32) m = pk_max_i(m, dppu<0x4E>(m));
  if (gs >= 64) m = pk_max_i(m, dppu<0x141>(m));
  if (gs >= 128) m = pk_max_i(m, dppu<0x140>(m));
  return m;
}

__device__ __forceinline__ float half_bits(uint32_t b) {
  return (float)__builtin_bit_cast(half_t, (uint16_t)b);
}
// token of a tile that lane group g loads as its i-th: four whole rows an instruction; in the
// TILE32 order the 8 tokens of a lane are those of its 32 bytes (tile32_offset)
template <bool TILE>
__device__ __forceinline__ constexpr int tok_of_i(int i) {
  return TILE ? 16 * (i >> 2) + (i & 3) : 4 * i;
}
// a lane's 8 channels of a row; a side with outlier channels reads single values of the row
// again, so its rows stay in the caches (streamed, they were fetched twice: 171 -> 131 us at
// 8 x 4 heads x 32768 tokens)
enum RowLoad { kStream, kCached, kDwords };  // kDwords: rows aligned to 4 bytes only
template <RowLoad LD>
__device__ __forceinline__ u32x4 ld_row(const half_t* p) {
  if constexpr (LD == kDwords) {
    const uint32_t* q = reinterpret_cast<const uint32_t*>(p);
    return u32x4{q[0], q[1], q[2], q[3]};
  }
  const u32x4* q = reinterpret_cast<const u32x4*>(p);
  if constexpr (LD == kStream) return __builtin_nontemporal_load(q);
  return *q;
}
template <bool TILE>
__device__ __forceinline__ int tok_of_g(int g) {
  return TILE ? 4 * g : g;
}

// a lane's rows of the tile at prompt token s0; rows outside the prompt read its first / last row
template <int NT, bool TILE, RowLoad LD>
__device__ __forceinline__ void load_tile(const AppendDev& a, const half_t* xr, int s0, int g, int d0,
                                          bool full, u32x4 w[NT]) {
  if (full) {  // lane base + uniform offsets
    const half_t* xl = xr + (int64_t)(s0 + tok_of_g<TILE>(g)) * a.xss + d0;
#pragma unroll
    for (int i = 0; i < NT; ++i) w[i] = ld_row<LD>(xl + tok_of_i<TILE>(i) * a.xss);
  } else {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int s = min(max(s0 + tok_of_g<TILE>(g) + tok_of_i<TILE>(i), 0), a.S - 1);
      w[i] = ld_row<LD>(xr + (int64_t)s * a.xss + d0);
    }
  }
}

// ---------------------------------------------------------------- INT4 group rescue
//
// The threshold is torch.quantile over the dynamic scales fmax(absmax, 1e-5) / 7 of every
// (row, group) of the append (src/cache/int4_cache.py:384-390).  The scale is a non-decreasing
// function of the group's fp16 absmax, so its order statistics are those of the absmax's 15 bits:
// a histogram of the upper 8 bits finds the buckets of both ranks, a second one the lower 7 bits
// in each.  A NaN counts as 0, as fmaxf drops it.  (At 2 x 4 heads x 4096 tokens in groups of 16
// the append took 888 us with four 8-bit passes over the fp32 scales and a counting pass per
// side, 344 us with the tile kernel behind them, 35 us with these.)

__device__ __forceinline__ float rescue_scale(uint32_t key) {
  return __fdiv_rn(fmaxf(half_bits(key), 1e-5f), 7.0f);
}

// f(key) for the absmax key of each (row, group) of the tile's valid rows, one lane a group (i: the
// lane's row of the tile)
template <int NT, class F>
__device__ __forceinline__ void tile_keys(const AppendDev& a, const u32x4 w[NT], int s0, int g, int c, F f) {
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    uint32_t k[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      k[j] = w[i][j] & 0x7FFF7FFFu;
      if ((k[j] & 0xFFFFu) > 0x7C00u) k[j] &= 0xFFFF0000u;
      if ((k[j] >> 16) > 0x7C00u) k[j] &= 0xFFFFu;
    }
    uint32_t m = pk_max_i(pk_max_i(k[0], k[1]), pk_max_i(k[2], k[3]));
    m = max_group(pk_max_i(m, swap16(m)), a.gs) & 0xFFFFu;
    const int s = s0 + 4 * i + g;
    if (s < a.S && (8 * c) % a.gs == 0) f(i, m);
  }
}

// The bin of h[0, n) (n = 64 R bins from h, R a lane) that holds rank r, and r's rank within it;
// one wave, every lane gets the result.
template <int R>
__device__ __forceinline__ void bin_of_rank(const uint32_t* h, uint32_t r, int lane, uint32_t& bin,
                                            uint32_t& within) {
  uint32_t v[R], sum = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) sum += v[i] = h[R * lane + i];
  // inclusive prefix sum over the wave: within rows of 16 by DPP, then the row totals
  uint32_t upto = sum;
  upto += dpp_shr<0x111>(upto);  // row_shr:1
  upto += dpp_shr<0x112>(upto);
  upto += dpp_shr<0x114>(upto);
  upto += dpp_shr<0x118>(upto);
  const uint32_t r0 = __builtin_amdgcn_readlane(upto, 15), r1 = r0 + __builtin_amdgcn_readlane(upto, 31),
                 r2 = r1 + __builtin_amdgcn_readlane(upto, 47);
  upto += lane < 16 ? 0u : lane < 32 ? r0 : lane < 48 ? r1 : r2;
  const uint64_t past = __ballot(r < upto);  // lanes whose bins reach past r
  const int owner = past ? __builtin_ctzll(past) : 63;
  uint32_t cum = upto - sum, b = R * lane, at = 0;
  bool found = false;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (!found && r < cum + v[i]) {
      b = R * lane + i;
      at = r - cum;
      found = true;
    }
    cum += v[i];
  }
  bin = __builtin_amdgcn_readlane(b, owner);
  within = __builtin_amdgcn_readlane(at, owner);
}

// rank of torch.quantile's lower order statistic: lo = floor(fp32(q) * (n - 1)); hi = ceil
__device__ __forceinline__ void quantile_ranks(float q, int64_t n, uint32_t& lo, uint32_t& hi, float& w) {
  const float rank = q * (float)(n - 1);
  const float f = floorf(rank);
  lo = (uint32_t)f;
  hi = (uint32_t)ceilf(rank);
  w = rank - f;
}

// The select's state of one side, in the caller's scratch: the histogram of the upper 8 bits,
// then (cleared by rescue_bucket_kernel) those of the lower 7 bits in the buckets of both ranks.
struct RescueScratch {
  uint32_t hist[256];
  uint32_t bucket[2];  // upper bits of sorted[lo], sorted[hi]
  uint32_t rank[2];    // their ranks within the buckets
  uint32_t pad[4];
};

__device__ __forceinline__ RescueScratch* scratch_of(const AppendDev& a) {
  return reinterpret_cast<RescueScratch*>(a.rescue);
}

// the threshold from the lower-bit histograms; one wave
__device__ __forceinline__ float rescue_threshold(const AppendDev& a, const uint32_t* hist,
                                                  const uint32_t* bucket, const uint32_t* rank, int lane) {
  uint32_t lo, hi, k0, k1, at;
  float w;
  quantile_ranks(a.rq, (int64_t)a.B * a.H * a.S * (128 / a.gs), lo, hi, w);
  bin_of_rank<2>(hist, rank[0], lane, k0, at);
  bin_of_rank<2>(hist + 128, rank[1], lane, k1, at);
  return quantile_lerp(rescue_scale(bucket[0] << 7 | k0), rescue_scale(bucket[1] << 7 | k1), w);
}

}  // namespace

}  // namespace kvq
