// Dequantised fp16 K / V of a cache layer (the engines' get_kv).
//
// What bounds it: HBM, mostly the fp16 rows written (256 of 320 to 400 bytes per token and head).
// One launch does both sides: a wave takes 16 (8) tokens of one (b, head), lane (g, c) channels
// 8 c .. 8 c + 7 of every fourth, so codes are read and fp16 rows written four whole rows an
// instruction.  INT4 in groups of 32, 8 x 4 heads x 32768 tokens (705 MB): 118 us, 6.0 TB/s;
// 2 x 4 x 6001: 8.5 us, where torch's unpack, cast, multiply and cast took 165 us in about 14
// passes a side.  The arithmetic is the engines' torch expressions', rounded where they
// round: a symmetric side fp16(c s) with the product in fp32 (an fp16 scale's product is exact
// there, so this is torch's fp16 product too), an asymmetric one fp16(c s + z) with product and
// sum rounded to fp32 each.
#include "append_tile.h"
#include "engine_ops.h"

#pragma clang fp contract(off)

namespace kvq {

namespace {

constexpr int kDeqWaves = 4;

struct DeqSide {
  int fmt, gs;
  const uint8_t* codes;
  int64_t sb, sh, st;
  const void* scale;
  const float* zp;
  int64_t ssb, ssh, sst, ssg;
  int scale_f32, per_channel;
  half_t* out;  // [B, H, n, 128] dense
};

// R: rows a lane holds (4 R tokens a wave)
template <bool I4, bool ASYM, int R>
__device__ __forceinline__ void deq_side(const DeqSide& a, int B, int H, int n) {
  constexpr int kTokens = 4 * R;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15, ntile = (n + kTokens - 1) / kTokens;
  const int items = B * H * ntile;
  for (int item = blockIdx.x * kDeqWaves + wave; item < items; item += gridDim.x * kDeqWaves) {
    const int bh = item / ntile, b = bh / H, h = bh - b * H, t0 = (item - bh * ntile) * kTokens + g;
    const uint8_t* cp = a.codes + (int64_t)b * a.sb + (int64_t)h * a.sh + (I4 ? 4 : 8) * c;
    half_t* const o = a.out + ((int64_t)bh * n + t0) * 128 + 8 * c;
    uint32_t w[R][I4 ? 1 : 2];
    float s[R], z[R], sc[8], zc[8];
    const int64_t so = (int64_t)b * a.ssb + (int64_t)h * a.ssh + (ASYM ? 0 : (int64_t)(8 * c / a.gs) * a.ssg);
    if (ASYM && a.per_channel) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sc[j] = reinterpret_cast<const float*>(a.scale)[so + 8 * c + j];
        zc[j] = a.zp[so + 8 * c + j];
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t t = min(t0 + 4 * i, n - 1);
      const uint8_t* p = cp + t * a.st;
      if constexpr (I4) {
        w[i][0] = ld_stream<uint32_t>(p);
      } else {
        const u32x2 v = ld_stream<u32x2>(p);
        w[i][0] = v.x;
        w[i][1] = v.y;
      }
      if (ASYM && a.per_channel) continue;
      const int64_t off = so + t * a.sst;
      s[i] = a.scale_f32 ? reinterpret_cast<const float*>(a.scale)[off]
                         : (float)reinterpret_cast<const half_t*>(a.scale)[off];
      if constexpr (ASYM) z[i] = a.zp[off];
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      float q[8];
      if constexpr (I4) {  // byte k: channels 2 k (high nibble), 2 k + 1, offset 8
        const uint32_t e = (w[i][0] >> 4) & 0x0F0F0F0Fu, d = w[i][0] & 0x0F0F0F0Fu;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          q[2 * k] = (float)((e >> (8 * k)) & 255u) - 8.0f;
          q[2 * k + 1] = (float)((d >> (8 * k)) & 255u) - 8.0f;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = (float)(int)(int8_t)(w[i][j >> 2] >> (8 * (j & 3)));
      }
      uint32_t r[4];
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        half2v v;
        if constexpr (ASYM) {
          const bool pc = a.per_channel;
          const float p0 = q[j] * (pc ? sc[j] : s[i]), p1 = q[j + 1] * (pc ? sc[j + 1] : s[i]);
          v = half2v{(half_t)(p0 + (pc ? zc[j] : z[i])), (half_t)(p1 + (pc ? zc[j + 1] : z[i]))};
        } else {
          v = half2v{(half_t)(q[j] * s[i]), (half_t)(q[j + 1] * s[i])};
        }
        r[j >> 1] = as_u32(v);
      }
      if (t0 + 4 * i < n)
        __builtin_nontemporal_store(u32x4{r[0], r[1], r[2], r[3]}, reinterpret_cast<u32x4*>(o + i * 512));
    }
  }
}

template <int FMT, int R>
__device__ __forceinline__ void deq(const DeqSide& a, int B, int H, int n) {
  if (!a.codes) return;
  deq_side<FMT == KVQ_FMT_INT4_SYM || FMT == KVQ_FMT_INT4_KIVI,
           FMT == KVQ_FMT_INT4_KIVI || FMT == KVQ_FMT_INT8_KIVI, R>(a, B, H, n);
}

// FK / FV: the formats of K and V (a missing side has the other one's); grid.y selects the side
template <int FK, int FV, int R>
__global__ __launch_bounds__(kDeqWaves * 64) void dequant_kernel(DeqSide k, DeqSide v, int B, int H, int n) {
  if (blockIdx.y == 0) deq<FK, R>(k, B, H, n);
  else deq<FV, R>(v, B, H, n);
}

template <int FK, int FV>
void go(const DeqSide& k, const DeqSide& v, int B, int H, int n, hipStream_t st) {
  // rows in flight a lane: an asymmetric side's parameters take the registers of two (8 x 4 heads x
  // 32768 tokens, us for 2 / 4 / 8: INT4 119 / 118 / 116, INT8 139 / 134 / 141, KIVI INT4 138 / 164
  // / 209)
  constexpr bool asym = FK == KVQ_FMT_INT4_KIVI || FK == KVQ_FMT_INT8_KIVI || FV == KVQ_FMT_INT4_KIVI ||
                        FV == KVQ_FMT_INT8_KIVI;
  constexpr int R = asym ? 2 : 4;
  const int64_t tiles = (int64_t)B * H * (((int64_t)n + 4 * R - 1) / (4 * R));
  int64_t gx = (tiles + kDeqWaves - 1) / kDeqWaves;
  if (gx > 65535) gx = 65535;
  hipLaunchKernelGGL((dequant_kernel<FK, FV, R>), dim3((unsigned)gx, 2), dim3(kDeqWaves * 64), 0, st, k, v,
                     B, H, n);
}

// the launch of a pair of formats (those the engines form), or nullptr
using Launch = void (*)(const DeqSide&, const DeqSide&, int, int, int, hipStream_t);
Launch pick(int fk, int fv) {
#define KVQ_DEQ(A, B) if (fk == A && fv == B) return go<A, B>
  KVQ_DEQ(KVQ_FMT_INT8_SYM, KVQ_FMT_INT8_SYM);
  KVQ_DEQ(KVQ_FMT_INT4_SYM, KVQ_FMT_INT4_SYM);
  KVQ_DEQ(KVQ_FMT_INT4_KIVI, KVQ_FMT_INT4_KIVI);
  KVQ_DEQ(KVQ_FMT_INT4_KIVI, KVQ_FMT_INT8_KIVI);
  KVQ_DEQ(KVQ_FMT_INT8_KIVI, KVQ_FMT_INT4_KIVI);
  KVQ_DEQ(KVQ_FMT_INT8_KIVI, KVQ_FMT_INT8_KIVI);
  KVQ_DEQ(KVQ_FMT_INT8_SYM, KVQ_FMT_INT4_KIVI);
  KVQ_DEQ(KVQ_FMT_INT4_KIVI, KVQ_FMT_INT8_SYM);
#undef KVQ_DEQ
  return nullptr;
}

int fill_side(const kvq_kv_view* x, int32_t fmt, int32_t gs, void* out, DeqSide& d, const char* name) {
  d = DeqSide{};
  if (!x) return KVQ_OK;
  const std::string n(name);
  const bool i4 = fmt == KVQ_FMT_INT4_SYM || fmt == KVQ_FMT_INT4_KIVI;
  const bool asym = fmt == KVQ_FMT_INT4_KIVI || fmt == KVQ_FMT_INT8_KIVI;
  if (!i4 && fmt != KVQ_FMT_INT8_SYM && fmt != KVQ_FMT_INT8_KIVI)
    return fail(KVQ_ERR_UNSUPPORTED, n + ": no dequantiser for this format");
  if (!x->codes || !x->scale || !out || (asym && !x->zero_point))
    return fail(KVQ_ERR_INVALID, n + ": NULL pointer");
  const int unit = i4 ? 4 : 8;
  if ((uintptr_t)x->codes % unit || x->stride_b % unit || x->stride_h % unit || x->stride_t % unit ||
      (uintptr_t)out % 16)
    return fail(KVQ_ERR_UNSUPPORTED, n + ": rows must be aligned");
  if (asym ? x->scale_dtype != KVQ_DTYPE_F32
           : (gs != 8 && gs != 16 && gs != 32 && gs != 64 && gs != 128))
    return fail(KVQ_ERR_UNSUPPORTED, n + ": scales");
  d.fmt = fmt;
  d.gs = gs;
  d.codes = reinterpret_cast<const uint8_t*>(x->codes);
  d.sb = x->stride_b; d.sh = x->stride_h; d.st = x->stride_t;
  d.scale = x->scale;
  d.zp = reinterpret_cast<const float*>(x->zero_point);
  d.ssb = x->scale_stride_b; d.ssh = x->scale_stride_h; d.sst = x->scale_stride_t; d.ssg = x->scale_stride_g;
  d.scale_f32 = x->scale_dtype == KVQ_DTYPE_F32;
  d.per_channel = asym && x->scale_stride_g == 1;
  d.out = reinterpret_cast<half_t*>(out);
  return KVQ_OK;
}

}  // namespace

}  // namespace kvq

using namespace kvq;

extern "C" int kvq_dequant(const kvq_kv_view* k, int32_t k_format, int32_t k_group, void* k_out,
                           const kvq_kv_view* v, int32_t v_format, int32_t v_group, void* v_out,
                           int32_t batch, int32_t heads, int32_t tokens, kvq_stream_t stream) {
  if (batch < 0 || heads < 0 || tokens < 0) return fail(KVQ_ERR_INVALID, "dequant: negative size");
  DeqSide dk, dv;
  int rc = fill_side(k, k_format, k_group, k_out, dk, "k");
  if (rc) return rc;
  if ((rc = fill_side(v, v_format, v_group, v_out, dv, "v"))) return rc;
  if ((int64_t)batch * heads * tokens > (1 << 30)) return fail(KVQ_ERR_UNSUPPORTED, "dequant: too many rows");
  if (!k && !v) return KVQ_OK;
  const Launch launch = pick(dk.codes ? dk.fmt : dv.fmt, dv.codes ? dv.fmt : dk.fmt);
  if (!launch) return fail(KVQ_ERR_UNSUPPORTED, "dequant: no kernel for this pair of formats");
  if ((int64_t)batch * heads * tokens == 0) return KVQ_OK;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  launch(dk, dv, batch, heads, tokens, st);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? KVQ_OK : fail(KVQ_ERR_LAUNCH, std::string("launch: ") + hipGetErrorString(e));
}
