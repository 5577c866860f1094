// Per-channel ranges of a prompt's K (the frozen parameters of the KIVI layout).
//
// Percentiles, and min / max up to range_splits: one work-group takes 8 channels of one (b, head)
// over all tokens, so nothing is merged between work-groups and the whole reduction is one launch: a
// thread reads 16 bytes of a token's row.
// The 16 work-groups of a (b, head) run on one XCD (work-group ids go round the 8 XCDs), whose L2
// then fetches each row once for all of them.
//
// Percentiles are exact order statistics by radix select: fp16 values as 16-bit integers in their
// order, a histogram of the upper byte per channel finds the byte of each of the four ranks, a
// second one the lower byte of the values in those buckets (few: the ranks lie in the tails).
// Up to kRows rows a thread stay in registers for the second pass; longer prompts are read
// again (L2, or the Infinity Cache).
//
// Bound: few units leave CUs idle, and a CU takes about two cycles for the 128-byte line of every
// row (1 x 2 heads x 32768 tokens: 40 us for min / max, why long prompts split it); then the LDS
// atomics of the first histogram.  4 heads x 1999 tokens: min / max 4.8 us (torch's aminmax of the
// fp32 copy 48 us); 4 x 8191: 99.9 percentiles 20.7 us (torch.sort in fp32 with index arrays,
// transposes and casts about 300 us); 8 x 4 heads x 32768: 178 us, min / max 48 us (5.6 TB/s).
#include "append_tile.h"
#include "engine_ops.h"

#pragma clang fp contract(off)

namespace kvq {

namespace {

constexpr int kRows = 8;    // rows a thread holds
constexpr int kCopies = 4;  // copies of the upper-byte histogram: the values crowd in a few bins
constexpr int kStride = 257;
constexpr int kSplitGroups = 2048;  // work-groups of the split min / max: 8 of 256 threads a CU

struct RangeArgs {
  const half_t* x;
  int64_t sb, sh, ss;
  int H, S, units;  // units = B * H
  int first;        // the launch's first unit (launch_range)
  float qmin, span;
  int r[4];         // ranks: lower tail floor / ceil, upper tail floor / ceil
  float wl, wh;
  float *scale, *zp;
  uint32_t* part;   // min / max by splits: [units, splits, 2, 64] packed keys
  int splits;
};

// fp16 bits -> 16-bit unsigned keys in the order of the values, every NaN above them all
__device__ __forceinline__ uint32_t key2(uint32_t w) {
  const i16x2 v = __builtin_bit_cast(i16x2, w);
  const uint32_t s = __builtin_bit_cast(uint32_t, v >> 15);
  uint32_t k = w ^ (s | 0x80008000u);
  if ((w & 0x7FFFu) > 0x7C00u) k |= 0xFFFFu;
  if ((w & 0x7FFF0000u) > 0x7C000000u) k |= 0xFFFF0000u;
  return k;
}
__device__ __forceinline__ float value_of(uint32_t key) {
  return half_bits(key & 0x8000u ? key ^ 0x8000u : key ^ 0xFFFFu);
}

template <RowLoad LD>
__device__ __forceinline__ void load_rows(const RangeArgs& a, const half_t* xr, int s0, u32x4 w[kRows]) {
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int s = min(s0 + i * (int)blockDim.x + (int)threadIdx.x, a.S - 1);
    w[i] = ld_row<LD>(xr + (int64_t)s * a.ss);
  }
}

// s, z of one channel (torch.clamp keeps a NaN range)
__device__ __forceinline__ void store_range(const RangeArgs& a, int64_t at, float mn, float mx) {
  const float floor = fmaxf(1e-5f, 6.103515625e-05f * a.span);
  float range = mx - mn;
  if (range < floor) range = floor;
  const float s = __fdiv_rn(range, a.span);
  a.scale[at] = s;
  a.zp[at] = mn - a.qmin * s;
}

template <bool PCT, RowLoad LD>
__global__ __launch_bounds__(1024) void kivi_range_kernel(RangeArgs a) {
  // 128 consecutive work-groups: 8 units (one an XCD) x 16 channel slices
  const int slice = (blockIdx.x >> 3) & 15, unit = a.first + (blockIdx.x & 7) + 8 * (blockIdx.x >> 7);
  if (unit >= a.units) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6, span = kRows * blockDim.x;
  const half_t* xr = a.x + (int64_t)(unit / a.H) * a.sb + (int64_t)(unit % a.H) * a.sh + 8 * slice;
  const int64_t out = (int64_t)unit * 128 + 8 * slice;
  u32x4 w[kRows];

  if constexpr (!PCT) {
    __shared__ uint32_t red[16][8];
    uint32_t hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};  // largest key and largest ~key
    for (int s0 = 0; s0 < a.S; s0 += span) {
      load_rows<LD>(a, xr, s0, w);  // rows past the end repeat the last one
#pragma unroll
      for (int i = 0; i < kRows; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t k = key2(w[i][j]);
          hi[j] = pk_max_u(hi[j], k);
          lo[j] = pk_max_u(lo[j], ~k);
        }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        hi[j] = pk_max_u(hi[j], (uint32_t)__shfl_xor((int)hi[j], o, 64));
        lo[j] = pk_max_u(lo[j], (uint32_t)__shfl_xor((int)lo[j], o, 64));
      }
    if (lane == 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[wave][j] = hi[j], red[wave][4 + j] = lo[j];
    __syncthreads();
    if (threadIdx.x < 8) {
      const int j = threadIdx.x >> 1, sft = 16 * (threadIdx.x & 1);
      uint32_t h = 0, l = 0;
      for (int i = 0; i < waves; ++i) {
        h = max(h, (red[i][j] >> sft) & 0xFFFFu);
        l = max(l, (red[i][4 + j] >> sft) & 0xFFFFu);
      }
      const float mx = value_of(h);
      // a NaN makes both ends NaN, as torch.aminmax
      store_range(a, out + threadIdx.x, h == 0xFFFFu ? mx : value_of(~l & 0xFFFFu), mx);
    }
  } else {
    // upper-byte histograms in kCopies copies, then (same memory) the four buckets' lower bytes
    __shared__ uint32_t h[8 * 4 * kStride];
    static_assert(kCopies == 4, "the two uses have the same size");
    __shared__ uint32_t upper[8][4], rank[8][4], lower[8][4];
    for (int i = threadIdx.x; i < 8 * 4 * kStride; i += blockDim.x) h[i] = 0;
    __syncthreads();
    uint32_t* const mine = h + (lane & 3) * kStride;
    for (int s0 = 0; s0 < a.S; s0 += span) {
      load_rows<LD>(a, xr, s0, w);
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        if (s0 + i * (int)blockDim.x + (int)threadIdx.x >= a.S) break;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t k = key2(w[i][j]);
          atomicAdd(&mine[(2 * j) * 4 * kStride + ((k >> 8) & 255u)], 1u);
          atomicAdd(&mine[(2 * j + 1) * 4 * kStride + (k >> 24)], 1u);
        }
      }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 8 * 256; i += blockDim.x) {
      uint32_t* const c = h + (i >> 8) * 4 * kStride + (i & 255);
      c[0] += c[kStride] + c[2 * kStride] + c[3 * kStride];
    }
    __syncthreads();
    for (int i = wave; i < 32; i += waves) {
      uint32_t b, at;
      bin_of_rank<4>(h + (i >> 2) * 4 * kStride, (uint32_t)a.r[i & 3], lane, b, at);
      if (lane == 0) upper[i >> 2][i & 3] = b, rank[i >> 2][i & 3] = at;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 8 * 4 * kStride; i += blockDim.x) h[i] = 0;
    uint32_t low[8], high[8];  // a value below / above these bytes' buckets is in no tail
#pragma unroll
    for (int j = 0; j < 8; ++j) low[j] = upper[j][1], high[j] = upper[j][2];
    __syncthreads();
    for (int s0 = 0; s0 < a.S; s0 += span) {
      if (a.S > span) load_rows<LD>(a, xr, s0, w);
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        if (s0 + i * (int)blockDim.x + (int)threadIdx.x >= a.S) break;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t k = (key2(w[i][j >> 1]) >> (16 * (j & 1))) & 0xFFFFu, ub = k >> 8;
          if (ub > low[j] && ub < high[j]) continue;
#pragma unroll
          for (int t = 0; t < 4; ++t)
            if (ub == upper[j][t]) atomicAdd(&h[(j * 4 + t) * kStride + (k & 255u)], 1u);
        }
      }
    }
    __syncthreads();
    for (int i = wave; i < 32; i += waves) {
      uint32_t b, at;
      bin_of_rank<4>(h + i * kStride, rank[i >> 2][i & 3], lane, b, at);
      if (lane == 0) lower[i >> 2][i & 3] = b;
    }
    __syncthreads();
    if (threadIdx.x < 8) {
      float v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) v[t] = value_of(upper[threadIdx.x][t] << 8 | lower[threadIdx.x][t]);
      store_range(a, out + threadIdx.x, quantile_lerp(v[0], v[1], a.wl), quantile_lerp(v[2], v[3], a.wh));
    }
  }
}

// Min / max of a long prompt in two launches: work-groups of whole rows over all CUs (a wave reads
// four rows an instruction), each leaving the largest keys and largest ~keys of its tokens, then
// one work-group a unit over those.  Bound: the rows' bytes, plus the second launch (about 4 us).
template <RowLoad LD>
__global__ __launch_bounds__(256) void kivi_range_part_kernel(RangeArgs a) {
  const int split = (int)blockIdx.x % a.splits, unit = (int)blockIdx.x / a.splits;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = threadIdx.x & 15;
  const int chunk = ((a.S + a.splits - 1) / a.splits + 127) / 128 * 128;  // tokens of a work-group
  const int end = min(a.S, (split + 1) * chunk);
  const half_t* xr = a.x + (int64_t)(unit / a.H) * a.sb + (int64_t)(unit % a.H) * a.sh + 8 * c;
  __shared__ uint32_t red[4][2][64];
  uint32_t hi[4] = {0, 0, 0, 0}, lo[4] = {0, 0, 0, 0};  // (an empty split leaves these)
  for (int s0 = split * chunk; s0 < end; s0 += 128) {
    u32x4 w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)  // rows past the end repeat the last one
      w[i] = ld_row<LD>(xr + (int64_t)min(s0 + 16 * i + (int)(threadIdx.x >> 4), end - 1) * a.ss);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t k = key2(w[i][j]);
        hi[j] = pk_max_u(hi[j], k);
        lo[j] = pk_max_u(lo[j], ~k);
      }
  }
#pragma unroll
  for (int o = 16; o < 64; o <<= 1)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      hi[j] = pk_max_u(hi[j], (uint32_t)__shfl_xor((int)hi[j], o, 64));
      lo[j] = pk_max_u(lo[j], (uint32_t)__shfl_xor((int)lo[j], o, 64));
    }
  if (lane < 16)
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave][0][4 * c + j] = hi[j], red[wave][1][4 * c + j] = lo[j];
  __syncthreads();
  if (threadIdx.x < 128) {
    const uint32_t* r = &red[0][0][threadIdx.x];
    a.part[(int64_t)blockIdx.x * 128 + threadIdx.x] =
        pk_max_u(pk_max_u(r[0], r[128]), pk_max_u(r[256], r[384]));
  }
}

__global__ __launch_bounds__(1024) void kivi_range_merge_kernel(RangeArgs a) {
  const int unit = blockIdx.x, col = threadIdx.x & 127, grp = threadIdx.x >> 7;
  const uint32_t* p = a.part + (int64_t)unit * a.splits * 128 + col;
  __shared__ uint32_t red[8][128];
  uint32_t m = 0;
  for (int i = grp; i < a.splits; i += 8) m = pk_max_u(m, p[(int64_t)i * 128]);
  red[grp][col] = m;
  __syncthreads();
  if (threadIdx.x < 128) {
    const int pair = threadIdx.x >> 1, sft = 16 * (threadIdx.x & 1);
    uint32_t h = 0, l = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      h = max(h, (red[i][pair] >> sft) & 0xFFFFu);
      l = max(l, (red[i][64 + pair] >> sft) & 0xFFFFu);
    }
    const float mx = value_of(h);
    store_range(a, (int64_t)unit * 128 + threadIdx.x, h == 0xFFFFu ? mx : value_of(~l & 0xFFFFu), mx);
  }
}

// Work-groups a unit of the split min / max, or 0 for the single launch.  One launch against two, us:
// 1 x 2 heads x 1024 tokens 4.5 / 6.4, 1 x 4 x 1999 4.8 / 6.4, 1 x 2 x 4096 7.7 / 6.6 (a second
// launch also costs the host about 4), 1 x 4 x 8191 9.8 / 7.2, 8 x 8 x 1024 9.0 / 7.3, 4 x 8 x 4096
// 15.6 / 9.4, 1 x 2 x 32768 39.7 / 10.8, 8 x 8 x 8192 46.7 / 26.7, 8 x 4 x 32768 84.2 / 47.8: it pays
// where a unit's 16 CUs read long, or where the units' rows are many.
int range_splits(int64_t units, int tokens) {
  if (units <= 0 || tokens > (1 << 30)) return 0;
  if (tokens <= 8192 && (tokens < 1024 || units * tokens < 65536)) return 0;
  const int64_t most = ((int64_t)tokens + 255) / 256, fill = (kSplitGroups + units - 1) / units;
  return (int)(fill < most ? fill : most);
}

// A launch has fewer than 2^32 threads, and a unit is 16 work-groups of up to 1024.
constexpr int kLaunchUnits = 1 << 17;

template <bool PCT>
void launch_range(RangeArgs a, bool al16, hipStream_t st) {
  // 4 waves hold 2048 rows, 16 hold 8192; the percentiles' 64 selects want 16 waves at any length
  // (32 units of 333 tokens: 16.8 us with 4 waves and shuffled scans, 11.1 us)
  const dim3 block(!PCT && a.S <= kRows * 256 ? 256 : 1024);
  for (a.first = 0; a.first < a.units; a.first += kLaunchUnits) {
    const int n = a.units - a.first < kLaunchUnits ? a.units - a.first : kLaunchUnits;
    const dim3 grid((unsigned)((n + 7) / 8 * 128));
    if (al16) hipLaunchKernelGGL((kivi_range_kernel<PCT, kCached>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((kivi_range_kernel<PCT, kDwords>), grid, block, 0, st, a);
  }
}

}  // namespace

}  // namespace kvq

using namespace kvq;

extern "C" int64_t kvq_kivi_range_scratch_bytes(int32_t batch, int32_t heads, int32_t tokens, float q_hi) {
  const int64_t units = batch > 0 && heads > 0 ? (int64_t)batch * heads : 0;
  const int n = q_hi == 0.f ? range_splits(units, tokens) : 0;
  return n > 1 ? units * n * 128 * (int64_t)sizeof(uint32_t) : 0;
}

extern "C" int kvq_kivi_channel_range(const void* x, int64_t stride_b, int64_t stride_h, int64_t stride_s,
                                      int32_t batch, int32_t heads, int32_t tokens, int32_t bits, float q_lo,
                                      float q_hi, float* scale, float* zero_point, void* scratch,
                                      int64_t scratch_bytes, kvq_stream_t stream) {
  if (!x || !scale || !zero_point) return fail(KVQ_ERR_INVALID, "channel range: NULL pointer");
  if (batch < 0 || heads < 0 || tokens <= 0 || (int64_t)batch * heads > (1 << 30))
    return fail(KVQ_ERR_INVALID, "channel range: bad shape");
  if (bits != 4 && bits != 8) return fail(KVQ_ERR_INVALID, "channel range: bits must be 4 or 8");
  if (((uintptr_t)x % 4) || stride_b % 2 || stride_h % 2 || stride_s % 2)
    return fail(KVQ_ERR_UNSUPPORTED, "channel range: rows must be 4-byte aligned");
  // (a percentile just below 100 or above 50 rounds to the level 1 or to equal levels)
  if (!(q_hi == 0.f || (q_lo >= 0.f && q_lo <= q_hi && q_hi <= 1.f)))
    return fail(KVQ_ERR_INVALID, "channel range: quantile levels must lie in [0, 1]");
  if (batch * heads == 0) return KVQ_OK;
  RangeArgs a{};
  a.x = reinterpret_cast<const half_t*>(x);
  a.sb = stride_b; a.sh = stride_h; a.ss = stride_s;
  a.H = heads; a.S = tokens; a.units = batch * heads;
  a.qmin = bits == 4 ? -8.f : -128.f;
  a.span = bits == 4 ? 15.f : 255.f;
  a.scale = scale;
  a.zp = zero_point;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool al16 = (uintptr_t)x % 16 == 0 && stride_b % 8 == 0 && stride_h % 8 == 0 && stride_s % 8 == 0;
  if (q_hi == 0.f) {
    a.splits = range_splits(a.units, a.S);
    a.part = reinterpret_cast<uint32_t*>(scratch);
    if (a.splits > 1 && scratch && (uintptr_t)scratch % 4 == 0 &&
        scratch_bytes >= kvq_kivi_range_scratch_bytes(batch, heads, tokens, q_hi)) {
      const dim3 grid((unsigned)(a.units * a.splits));
      if (al16) hipLaunchKernelGGL((kivi_range_part_kernel<kCached>), grid, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((kivi_range_part_kernel<kDwords>), grid, dim3(256), 0, st, a);
      hipLaunchKernelGGL(kivi_range_merge_kernel, dim3((unsigned)a.units), dim3(1024), 0, st, a);
    } else {
      launch_range<false>(a, al16, st);
    }
  } else {
    // torch.quantile's fp32 ranks; ceil of a rank that rounded up to n - 1 stays in range
    const float n1 = (float)(tokens - 1), rl = q_lo * n1, rh = q_hi * n1;
    a.r[0] = (int)floorf(rl);
    a.r[1] = (int)ceilf(rl);
    a.r[2] = (int)floorf(rh);
    a.r[3] = (int)ceilf(rh);
    for (int& r : a.r) r = r > tokens - 1 ? tokens - 1 : r;
    a.wl = rl - (float)a.r[0];
    a.wh = rh - (float)a.r[2];
    launch_range<true>(a, al16, st);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? KVQ_OK : fail(KVQ_ERR_LAUNCH, std::string("launch: ") + hipGetErrorString(e));
}
