// Quantize-on-append of whole prompts: the append kernel's results (quant_append.hip), bit for
// bit, for rows that allow 16-byte loads and packed stores.
//
// What bounds it: HBM, with the quantizer's arithmetic not far behind (a wave64 VALU operation
// takes a SIMD about 1.7 ns and every value needs a correctly rounded division).  The row
// kernel gives a wave one row at a time, 4 bytes a lane, with single-byte stores into TILE32 and
// an atomic per row that clips: 0.63 TB/s at 8 x 4 heads x 32768 tokens of the asymmetric format
// (1069 us), 131 us (5.2 TB/s) here; with static INT8 tables at 4 x 8 x 16384 tokens 8254 -> 77 us
// (the atomics), INT8 with percentile scales at 2 x 4096 tokens 20.7 -> 5.4 us.
// Here a wave takes a tile of 32 tokens (8 where the prompt is short) of one (b, head): lane
// (g, c) holds channels 8 c .. 8 c + 7 of every fourth token, so a load instruction reads four
// whole rows, all of a tile's loads are in flight together, a group's statistics are DPP steps
// within 16 lanes and the codes leave as one store of 4, 8 or (TILE32) 16 bytes a lane.
//
// Divisions: q = RN(x / s) from the correctly rounded reciprocal r = RN(1 / s), which a static
// scale needs once per tile, by q = x r and two remainder corrections q += RN(x - q s) r (the
// remainder is a fused multiply-add; Markstein, "Computation of elementary functions on the IBM
// RISC System/6000", 1990: a faithful q corrected with a correctly rounded r is RN(x / s)).  It
// holds where nothing under- or overflows: tiles with a NaN or Inf, or a scale outside
// [2^-30, 2^30], are left to the row quantizer after the wave's other tiles.
#include "append_bulk.h"
#include "append_tile.h"
#include "engine_ops.h"

#pragma clang fp contract(off)

namespace kvq {

namespace {

// both halves shifted left by one (an fp16 value without its sign bit)
__device__ __forceinline__ uint32_t pk_double(uint32_t a) {
  const u16x2 v = __builtin_bit_cast(u16x2, a);
  return __builtin_bit_cast(uint32_t, (u16x2)(v + v));
}
// fp16 bits as signed 16-bit integers in the order of the values (-0 below +0), and back
__device__ __forceinline__ uint32_t sort_key2(uint32_t w) {
  const i16x2 v = __builtin_bit_cast(i16x2, w);
  const uint32_t s = __builtin_bit_cast(uint32_t, v >> 15);
  return w ^ (s & 0x7FFF7FFFu);
}
// The two largest 16-bit integers (with multiplicity) of a set, kept in both halves of m1 / m2.
struct Top2 {
  uint32_t m1, m2;
  __device__ __forceinline__ void merge(uint32_t n1, uint32_t n2) {
    m2 = pk_max_i(pk_min_i(m1, n1), pk_max_i(m2, n2));
    m1 = pk_max_i(m1, n1);
  }
};
__device__ __forceinline__ Top2 top2_of(const uint32_t k[4]) {
  Top2 t{pk_max_i(k[0], k[1]), pk_min_i(k[0], k[1])};
  t.merge(pk_max_i(k[2], k[3]), pk_min_i(k[2], k[3]));
  t.merge(swap16(t.m1), swap16(t.m2));
  return t;
}
// over the lanes of a group (gs / 8 consecutive lanes of 16); every lane gets the result
__device__ __forceinline__ void top2_group(Top2& t, int gs) {
  if (gs >= 16) t.merge(dppu<0xB1>(t.m1), dppu<0xB1>(t.m2));     // quad_perm [1, 0, 3, 2]
  if (gs >= 32) t.merge(dppu<0x4E>(t.m1), dppu<0x4E>(t.m2));     // quad_perm [2, 3, 0, 1]
  if (gs >= 64) t.merge(dppu<0x141>(t.m1), dppu<0x141>(t.m2));   // row_half_mirror
  if (gs >= 128) t.merge(dppu<0x140>(t.m1), dppu<0x140>(t.m2));  // row_mirror
}
// the value of a sort key (low half)
__device__ __forceinline__ float key_value(uint32_t k) {
  const int16_t v = (int16_t)k;
  return half_bits((uint32_t)(uint16_t)(v ^ ((v >> 15) & 0x7FFF)));
}

// RN(x / s) with r = RN(1 / s) (see the head of the file)
__device__ __forceinline__ float div_by(float x, float s, float r) {
  float q = x * r;
  q = fmaf(fmaf(-q, s, x), r, q);
  return fmaf(fmaf(-q, s, x), r, q);
}

// RN(1 / s): v_rcp_f32 and one fused correction, equal to the IEEE quotient for every significand
// (tests/test_gpu_append_division.py compares all 2^23 at eight exponents from -30 to 29; v_rcp_f32
// alone differs for 897,675 of them)
__device__ __forceinline__ float recip(float s) {
  const float r = __builtin_amdgcn_rcpf(s);
  return fmaf(fmaf(-s, r, 1.0f), r, r);
}

// the 8 values of a lane
struct Vals {
  float f[8];
};
__device__ __forceinline__ Vals vals(u32x4 w) {
  Vals v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const half2v h = as_h2(w[j]);
    v.f[2 * j] = (float)h.x;
    v.f[2 * j + 1] = (float)h.y;
  }
  return v;
}

// Low byte of each of 4 dwords -> one dword
__device__ __forceinline__ uint32_t bytes4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  const uint32_t ab = perm_b32(b, a, 0x0c0c0400u), cd = perm_b32(d, c, 0x0c0c0400u);
  return ab | (cd << 16);
}
// rint of a float in [-2^21, 2^21] plus off, as the low bits of a dword: adding 1.5 * 2^23 rounds
// to the nearest integer, ties to even (off is even)
__device__ __forceinline__ uint32_t rint_bits(float q, float off) {
  return __builtin_bit_cast(uint32_t, q + (12582912.0f + off));
}
__device__ __forceinline__ float clampf(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }

// 8 quotients -> 4 bytes of packed nibbles (even channel high, offset 8)
__device__ __forceinline__ uint32_t pack_nibbles(const float q[8], float lo, float hi) {
  uint32_t a[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t e = rint_bits(clampf(q[2 * j], lo, hi), 8.0f);
    const uint32_t o = rint_bits(clampf(q[2 * j + 1], lo, hi), 8.0f);
    a[j] = (e << 4) | o;  // low byte: o has nothing in bits 4..7
  }
  return bytes4(a[0], a[1], a[2], a[3]);
}
// 8 quotients -> 8 signed bytes
__device__ __forceinline__ u32x2 pack_bytes(const float q[8], float lo, float hi) {
  uint32_t a[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) a[j] = rint_bits(clampf(q[j], lo, hi), 0.0f);
  return u32x2{bytes4(a[0], a[1], a[2], a[3]), bytes4(a[4], a[5], a[6], a[7])};
}
// 8 quotients -> 8 INT8_SYM codes: rounded to fp16, clamped, rounded to integers (adding
// 1.5 * 2^10 in fp16), as bytes
__device__ __forceinline__ u32x2 pack_int8_sym(const float q[8]) {
  uint32_t a[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    half2v h = {(half_t)q[2 * j], (half_t)q[2 * j + 1]};
    h = __builtin_elementwise_min(__builtin_elementwise_max(h, half2v{(half_t)-127.f, (half_t)-127.f}),
                                  half2v{(half_t)127.f, (half_t)127.f});
    h += half2v{(half_t)1536.f, (half_t)1536.f};
    a[j] = as_u32(h);
  }
  return u32x2{perm_b32(a[1], a[0], 0x06040200u), perm_b32(a[3], a[2], 0x06040200u)};
}
// codes at +-127 among the 8 bytes
__device__ __forceinline__ int at_limit(u32x2 w) {
  int n = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int c = (int)(int8_t)(w[j >> 2] >> (8 * (j & 3)));
    n += (c == 127) | (c == -127);
  }
  return n;
}

// The threshold of a side of at most kRescueMax (row, group) scales, found by one work-group over
// all rows (each work-group of the append finds it itself).
struct LocalRescue {
  uint32_t hist[256], bucket[2], rank[2];
  uint16_t key[kRescueMax];
};
__device__ __forceinline__ float local_threshold(const AppendDev& a, LocalRescue& l) {
  constexpr int NT = 4, kTok = 4 * NT;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15, waves = blockDim.x >> 6, G = 128 / a.gs;
  const int rows = a.B * a.H * a.S, n = rows * G;
  for (int i = threadIdx.x; i < 256; i += blockDim.x) l.hist[i] = 0;
  __syncthreads();
  const int ntile = (a.S + kTok - 1) / kTok, items = a.B * a.H * ntile;
  for (int item = wave; item < items; item += waves) {
    const int bh = item / ntile, s0 = (item - bh * ntile) * kTok;
    const half_t* xr = a.x + (int64_t)(bh / a.H) * a.xsb + (int64_t)(bh % a.H) * a.xsh;
    u32x4 w[NT];
    load_tile<NT, false, kCached>(a, xr, s0, g, 8 * c, s0 + kTok <= a.S, w);
    tile_keys<NT>(a, w, s0, g, c, [&](int i, uint32_t key) {
      l.key[(bh * a.S + s0 + 4 * i + g) * G + 8 * c / a.gs] = (uint16_t)key;
      atomicAdd(&l.hist[key >> 7], 1u);
    });
  }
  __syncthreads();
  if (wave == 0) {
    uint32_t lo, hi, b, at;
    float w;
    quantile_ranks(a.rq, n, lo, hi, w);
    bin_of_rank<4>(l.hist, lo, lane, b, at);
    if (lane == 0) l.bucket[0] = b, l.rank[0] = at;
    bin_of_rank<4>(l.hist, hi, lane, b, at);
    if (lane == 0) l.bucket[1] = b, l.rank[1] = at;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += blockDim.x) l.hist[i] = 0;
  const uint32_t b0 = l.bucket[0], b1 = l.bucket[1];
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const uint32_t key = l.key[i];
    if (key >> 7 == b0) atomicAdd(&l.hist[key & 127], 1u);
    if (key >> 7 == b1) atomicAdd(&l.hist[128 + (key & 127)], 1u);
  }
  __syncthreads();
  return rescue_threshold(a, l.hist, l.bucket, l.rank, lane);
}

// One side of the append: FMT its format, NT tokens per lane (4 NT per tile), TILE the TILE32
// code layout.  Waves take tiles wave, wave + waves, ... (at most 64 each: `redo` has a bit per
// tile).
template <int FMT, int NT, bool TILE>
__device__ __forceinline__ void bulk_side(const AppendDev& a, const BulkSide& bs) {
  static_assert(!TILE || (FMT == KVQ_FMT_INT4_ASYM && NT == 8), "TILE32 tiles hold 32 tokens");
  constexpr int kTok = 4 * NT;
  constexpr bool kKivi = FMT == KVQ_FMT_INT4_KIVI || FMT == KVQ_FMT_INT8_KIVI;
  constexpr bool kSym = FMT == KVQ_FMT_INT4_SYM || FMT == KVQ_FMT_INT8_SYM;
  constexpr bool kByte = FMT == KVQ_FMT_INT8_SYM || FMT == KVQ_FMT_INT8_KIVI;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15, d0 = 8 * c;
  const int gs = a.gs, grp = d0 / gs;
  const int lead = TILE ? (int)(a.wpos & 31) : 0;  // slots of the first tile before the prompt
  const int ntile = (lead + a.S + kTok - 1) / kTok;
  const int waves = blockDim.x >> 6;
  const int items = a.B * a.H * ntile, step = gridDim.x * waves;
  float thr = 0.f;
  if constexpr (FMT == KVQ_FMT_INT4_SYM) {
    if (bs.local) {
      __shared__ LocalRescue local;
      thr = local_threshold(a, local);
    } else if (const RescueScratch* sc = scratch_of(a)) {
      thr = rescue_threshold(a, sc->hist, sc->bucket, sc->rank, lane);
    }
  }
  const bool table = a.st != nullptr;
  const bool outl = FMT == KVQ_FMT_INT4_ASYM && NT == 8 && a.n_out > 0;
  int clipped = 0;
  uint64_t redo = 0;
  int it = 0;
  for (int item = blockIdx.x * waves + wave; item < items; item += step, ++it) {
    const int bh = item / ntile, h = bh % a.H, b = bh / a.H;
    const int s0 = (item - bh * ntile) * kTok - lead;
    const half_t* xr = a.x + (int64_t)b * a.xsb + (int64_t)h * a.xsh;
    const bool full = s0 >= 0 && s0 + kTok <= a.S;
    u32x4 w[NT];
    if (outl) load_tile<NT, TILE, kCached>(a, xr, s0, g, d0, full, w);
    else load_tile<NT, TILE, kStream>(a, xr, s0, g, d0, full, w);
    // outlier channels (INT4_ASYM K): lane l copies channels 2 (l % 2), + 1 of token l / 2
    uint32_t ov = 0;
    const int so = s0 + (lane >> 1);
    if (outl) {
      const int2 oc = *reinterpret_cast<const int2*>(a.oidx + h * 4 + 2 * (lane & 1));
      const half_t* xo = xr + (int64_t)min(max(so, 0), a.S - 1) * a.xss;
      ov = as_u32(half2v{xo[min(max(oc.x, 0), 127)], xo[min(max(oc.y, 0), 127)]});
    }

    // the tile's fixed parameters
    float st = 0.f, sz = 0.f, ps[kKivi ? 8 : 1], pz[kKivi ? 8 : 1], pr[kKivi ? 8 : 1];
    bool bad = false;
    if constexpr (kSym) {
      if (table) {
        st = ld_static(a, h, grp);
        // INT8 rounds the scale to fp16; the adaptive product is the largest scale made of it
        const float top = a.adaptive ? fmaxf(st, 1e-5f) * a.margin : st;
        bad = !(top <= (FMT == KVQ_FMT_INT8_SYM ? 60000.0f : 1073741824.0f)) ||
              !(fabsf(st) <= 1073741824.0f);
        if constexpr (FMT == KVQ_FMT_INT8_SYM) {
          if (!a.adaptive) st = (float)int8_static_scale16(st, a.st_f32);
        }
      }
    } else if constexpr (FMT == KVQ_FMT_INT4_ASYM) {
      const int64_t off = (int64_t)h * a.st_sh + (int64_t)grp * a.st_sg;
      st = (float)reinterpret_cast<const half_t*>(a.st)[off];
      sz = (float)a.st_zp[off];
      bad = !(fabsf(st) > 0.f && fabsf(st) <= 65504.0f) || !(fabsf(sz) <= 65504.0f);
    } else if constexpr (kKivi) {
      if (table) {
        const int64_t o = (int64_t)b * a.st_sb + (int64_t)h * a.st_sh + d0;
        const float4* s4 = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(a.st) + o);
        const float4* z4 = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(a.st_zp) + o);
        const float4 sa = s4[0], sb = s4[1], za = z4[0], zb = z4[1];
        const float sv[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
        const float zv[8] = {za.x, za.y, za.z, za.w, zb.x, zb.y, zb.z, zb.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          ps[j] = sv[j];
          pz[j] = zv[j];
          pr[j] = recip(sv[j]);
          bad |= !(fabsf(sv[j]) >= 9.3132257e-10f && fabsf(sv[j]) <= 1073741824.0f) ||
                 !(fabsf(zv[j]) <= 1073741824.0f);
        }
      }
    }
    float rs = 0.f;  // reciprocal of a scale that is the same for every token
    if ((kSym && table && !a.adaptive && !bs.policy) || FMT == KVQ_FMT_INT4_ASYM) {
      if (FMT == KVQ_FMT_INT4_SYM) st = fmaxf(st, 1e-5f);
      rs = recip(st);
    }
    // NaN / Inf among the values: an exponent field of ones is at least 0xF800 without the sign
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        mx = pk_max_u(mx, pk_double(w[i][j]));
      }
    bad |= (mx >> 16) >= 0xF800u || (mx & 0xFFFFu) >= 0xF800u;
    if (__ballot(bad)) {
      redo |= 1ull << it;
      continue;
    }

    uint8_t* crow = a.codes + (int64_t)b * a.csb + (int64_t)h * a.csh;
    const int64_t srow = (int64_t)b * a.sosb + (int64_t)h * a.sosh;
    // the lane's first token; its i-th is tok_of_i(i) rows on
    const int64_t t0 = a.wpos + s0 + tok_of_g<TILE>(g);
    uint8_t* cl = crow + t0 * a.cst + (kByte ? d0 : 4 * c);
    const int64_t sl = srow + t0 * a.sost + (int64_t)grp * a.sosg;
    uint32_t tile[TILE ? NT : 1];
    float keep_s = 0.f, keep_z = 0.f;  // KIVI V: lane c keeps the parameters of its c-th token
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int s = s0 + tok_of_g<TILE>(g) + tok_of_i<TILE>(i);
      const bool in = full || (s >= 0 && s < a.S);
      uint8_t* const ct = cl + (int64_t)tok_of_i<TILE>(i) * a.cst;
      const Vals v = vals(w[i]);
      float q[8];
      if constexpr (FMT == KVQ_FMT_INT4_ASYM) {
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = div_by(v.f[j] - sz, st, rs);
        if (a.status) {
          int n = 0;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float r = rintf(q[j]);
            n += (r < -8.f) | (r > 7.f);
          }
          clipped += in ? n : 0;
        }
        const uint32_t codes = pack_nibbles(q, -8.f, 7.f);
        if constexpr (TILE) tile[i] = codes;
        else if (in) *reinterpret_cast<uint32_t*>(ct) = codes;
      } else if constexpr (kSym) {
        float sc = st, r = rs;
        bool over = table && a.status;  // whether the lane's group may hold clipped values
        if (!table || a.adaptive || bs.policy) {
          uint32_t k[4];  // |x| as integers (the values are finite)
#pragma unroll
          for (int j = 0; j < 4; ++j) k[j] = w[i][j] & 0x7FFF7FFFu;
          float am;
          if (!table && bs.top2) {
            Top2 m = top2_of(k);
            top2_group(m, gs);
            const float v1 = half_bits(m.m1), v2 = half_bits(m.m2);
            am = quantile_lerp(bs.lo == gs - 1 ? v1 : v2, bs.hi == gs - 1 ? v1 : v2, bs.w);
          } else {
            uint32_t m = pk_max_i(pk_max_i(k[0], k[1]), pk_max_i(k[2], k[3]));
            m = pk_max_i(m, swap16(m));
            am = half_bits(max_group(m, gs));
          }
          // the policies of int8_scale16 / int4_scale
          if (!table) {
            const float lo = bs.top2 ? 1e-5f : (float)(half_t)1e-5f;
            if constexpr (FMT == KVQ_FMT_INT8_SYM)
              sc = (float)(half_t)div_by((float)(half_t)fmaxf(am, lo), 127.0f, 1.0f / 127.0f);
            else
              sc = div_by(fmaxf(am, lo), 7.0f, 1.0f / 7.0f);
          } else if constexpr (FMT == KVQ_FMT_INT8_SYM) {
            sc = st;
            if (a.adaptive)
              sc = (float)(half_t)fmaxf(fmaxf(fmaxf(st, 1e-5f) * a.margin,
                                              div_by(fmaxf(am, 1e-5f), 127.0f, 1.0f / 127.0f)), 1e-5f);
          } else {
            const float dyn = div_by(fmaxf(am, 1e-5f), 7.0f, 1.0f / 7.0f);
            sc = fmaxf(st, 1e-5f);
            if (a.adaptive) sc = fmaxf(sc * a.margin, dyn);
            if (a.mixed || a.rescue_all || (a.rq > 0.f && dyn >= thr)) sc = fmaxf(sc, dyn);
            sc = fmaxf(sc, 1e-5f);
          }
          over = table && a.status && am > sc * (FMT == KVQ_FMT_INT8_SYM ? 126.0f : 7.0f);
          r = recip(sc);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = div_by(v.f[j], sc, r);
        if constexpr (FMT == KVQ_FMT_INT8_SYM) {
          const u32x2 codes = pack_int8_sym(q);
          if (over) clipped += in ? at_limit(codes) : 0;
          if (in) *reinterpret_cast<u32x2*>(ct) = codes;
        } else {
          if (over) {
            const float bound = sc * 7.0f;
            int n = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) n += fabsf(v.f[j]) > bound;
            clipped += in ? n : 0;
          }
          const uint32_t codes = pack_nibbles(q, -7.f, 7.f);
          if (in) *reinterpret_cast<uint32_t*>(ct) = codes;
        }
        if (a.so && in && d0 % gs == 0) {
          const int64_t off = sl + (int64_t)tok_of_i<TILE>(i) * a.sost;
          if (a.so_f32) reinterpret_cast<float*>(a.so)[off] = sc;
          else reinterpret_cast<half_t*>(a.so)[off] = (half_t)sc;
        }
      } else {  // KIVI
        constexpr bool b8 = FMT == KVQ_FMT_INT8_KIVI;
        constexpr float qmin = b8 ? -128.f : -8.f, qmax = b8 ? 127.f : 7.f, span = qmax - qmin;
        if (table) {
#pragma unroll
          for (int j = 0; j < 8; ++j) q[j] = div_by(v.f[j] - pz[j], ps[j], pr[j]);
          if (a.status) {
            int n = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) n += (q[j] < qmin) | (q[j] > qmax);
            clipped += in ? n : 0;
          }
        } else {
          uint32_t k[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) k[j] = sort_key2(w[i][j]);
          float mn, mx2;
          if (bs.top2) {
            Top2 hi = top2_of(k);
            top2_group(hi, 128);
            uint32_t nk[4];  // ~key orders the values downwards
#pragma unroll
            for (int j = 0; j < 4; ++j) nk[j] = ~k[j];
            Top2 lo = top2_of(nk);
            top2_group(lo, 128);
            const float h1 = key_value(hi.m1), h2 = key_value(hi.m2);
            const float l1 = key_value(~lo.m1), l2 = key_value(~lo.m2);
            mx2 = quantile_lerp(bs.lo == 127 ? h1 : h2, bs.hi == 127 ? h1 : h2, bs.w);
            mn = quantile_lerp(bs.blo == 0 ? l1 : l2, bs.bhi == 0 ? l1 : l2, bs.bw);
          } else {
            uint32_t m = pk_max_i(pk_max_i(k[0], k[1]), pk_max_i(k[2], k[3]));
            uint32_t n = pk_max_i(pk_max_i(~k[0], ~k[1]), pk_max_i(~k[2], ~k[3]));
            m = max_group(pk_max_i(m, swap16(m)), 128);
            n = max_group(pk_max_i(n, swap16(n)), 128);
            mx2 = key_value(m);
            mn = key_value(~n);
          }
          const float sc = div_by(fmaxf(mx2 - mn, span * 6.103515625e-05f), span, 1.0f / span);
          const float z = mn - qmin * sc;
          const float r = recip(sc);
          if (c == i) {
            keep_s = sc;
            keep_z = z;
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) q[j] = div_by(v.f[j] - z, sc, r);
        }
        if constexpr (b8) {
          const u32x2 codes = pack_bytes(q, qmin, qmax);
          if (in) *reinterpret_cast<u32x2*>(ct) = codes;
        } else {
          const uint32_t codes = pack_nibbles(q, qmin, qmax);
          if (in) *reinterpret_cast<uint32_t*>(ct) = codes;
        }
      }
    }
    if constexpr (kKivi) {
      if (!table && a.so && c < NT) {
        const int s = s0 + 4 * c + g;
        if (s < a.S) {
          const int64_t off = srow + (a.wpos + s) * a.sost;
          reinterpret_cast<float*>(a.so)[off] = keep_s;
          a.zo[off] = keep_z;
        }
      }
    }
    if constexpr (TILE) {
      // dword 2 p + k of the lane: bytes 2 k, 2 k + 1 of the two tokens (p, a = 0, 1)
      uint32_t o[8];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        o[2 * p] = perm_b32(tile[2 * p + 1], tile[2 * p], 0x05040100u);
        o[2 * p + 1] = perm_b32(tile[2 * p + 1], tile[2 * p], 0x07060302u);
      }
      uint8_t* ot = crow + ((a.wpos + s0) >> 5) * 2048 + 32 * lane;
      if (full) {
        reinterpret_cast<u32x4*>(ot)[0] = u32x4{o[0], o[1], o[2], o[3]};
        reinterpret_cast<u32x4*>(ot)[1] = u32x4{o[4], o[5], o[6], o[7]};
      } else {
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const int s = s0 + tok_of_g<TILE>(g) + tok_of_i<TILE>(i);
          if (s >= 0 && s < a.S) {
            uint16_t* p16 = reinterpret_cast<uint16_t*>(ot) + 4 * (i >> 1) + (i & 1);
            p16[0] = (uint16_t)tile[i];
            p16[2] = (uint16_t)(tile[i] >> 16);
          }
        }
      }
    }
    if (outl && so >= 0 && so < a.S)
      *reinterpret_cast<uint32_t*>(a.oo + (int64_t)b * a.oosb + (int64_t)h * a.oosh +
                                   (a.wpos + so) * a.oost + 2 * (lane & 1)) = ov;
  }
  // tiles left to the row quantizer
  while (redo) {
    const int i = __builtin_ctzll(redo);
    redo &= redo - 1;
    const int item = blockIdx.x * waves + wave + i * step;
    const int bh = item / ntile;
    const int s0 = (item - bh * ntile) * kTok - lead;
    for (int s = max(s0, 0); s < min(s0 + kTok, a.S); ++s) {
      const int row = bh * a.S + s;
      quant_row_x<FMT>(a, row, lane, thr, load_x(a, row, lane), row_static(a, row, lane));
    }
  }
  if (a.status) {
    __shared__ int cnt[kBulkMaxWaves];
    const int n = wave_sum_int(clipped);
    if (lane == 0) cnt[wave] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
      int sum = 0;
      for (int i = 0; i < waves; ++i) sum += cnt[i];
      if (sum) atomicAdd(&a.status[1], sum);
    }
  }
}

// FK / FV: the formats of K and V; grid.y selects the side
template <int FK, int FV, int NT, bool KT, bool VT>
__global__ __launch_bounds__(kBulkMaxWaves * 64) void append_bulk_kernel(AppendDev k, AppendDev v,
                                                                      BulkSide ks, BulkSide vs) {
  if (blockIdx.y == 0) {
    if (k.valid) bulk_side<FK, NT, KT>(k, ks);
  } else {
    if (v.valid) bulk_side<FV, NT, VT>(v, vs);
  }
}

__global__ void division_kernel(const float* x, const float* s, float* r, float* q, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  r[i] = recip(s[i]);
  q[i] = div_by(x[i], s[i], r[i]);
}

// the side's format, TILE32 apart from rows
constexpr int kTileAsym = 7;
int side_code(const AppendDev& d) { return d.tile32 ? kTileAsym : d.fmt; }

bool al(const void* p, int n) { return ((uintptr_t)p % n) == 0; }

// Whether the tile kernel takes side d: 16-byte aligned rows of x, code rows aligned to a lane's
// store, contiguous per-channel parameters, order statistics within the two largest (smallest).
bool side_ok(const AppendDev& d, BulkSide& s) {
  s = BulkSide{};
  if (!d.valid) return true;
  if (!al(d.x, 16) || d.xsb % 8 || d.xsh % 8 || d.xss % 8) return false;
  const int unit = d.tile32 ? 16 : (d.fmt == KVQ_FMT_INT8_SYM || d.fmt == KVQ_FMT_INT8_KIVI) ? 8 : 4;
  if (!al(d.codes, unit) || d.csb % unit || d.csh % unit || d.cst % unit) return false;
  const bool kivi = d.fmt == KVQ_FMT_INT4_KIVI || d.fmt == KVQ_FMT_INT8_KIVI;
  if (kivi && d.st != nullptr &&
      (d.st_sg != 1 || !al(d.st, 16) || !al(d.st_zp, 16) || d.st_sb % 4 || d.st_sh % 4))
    return false;
  if (d.n_out > 0 && (!al(d.oo, 4) || d.oosb % 2 || d.oosh % 2 || d.oost % 2 || !al(d.oidx, 8))) return false;
  s.policy = d.mixed || d.rescue_all || d.rq > 0.f;
  if (d.st == nullptr && d.dq > 0.f) {
    const int n = kivi ? 128 : d.gs;
    const float rank = d.dq * (float)(n - 1);
    s.lo = (int)floorf(rank);
    s.hi = (int)ceilf(rank);
    s.w = rank - (float)s.lo;
    s.top2 = 1;
    if (s.lo < n - 2 || s.hi > n - 1) return false;
    if (kivi) {
      const float low = d.dq_lo * (float)(n - 1);
      s.blo = (int)floorf(low);
      s.bhi = (int)ceilf(low);
      s.bw = low - (float)s.blo;
      if (s.bhi > 1) return false;
    }
  }
  return true;
}

template <int FK, int FV, int NT, bool KT = false, bool VT = false>
void go(const AppendDev& k, const AppendDev& v, const BulkPlan& p, hipStream_t st) {
  hipLaunchKernelGGL((append_bulk_kernel<FK, FV, NT, KT, VT>), dim3(p.groups, 2), dim3(p.waves * 64), 0, st, k,
                     v, p.ks, p.vs);
}

// the launch of a pair of side codes with tok tokens a wave, or nullptr
using Launch = void (*)(const AppendDev&, const AppendDev&, const BulkPlan&, hipStream_t);
Launch pick(int ck, int cv, int tok) {
#define KVQ_BULK(A, B) \
  if (ck == A && cv == B) return tok == 32 ? go<A, B, 8> : tok == 16 ? go<A, B, 4> : go<A, B, 2>
  KVQ_BULK(KVQ_FMT_INT8_SYM, KVQ_FMT_INT8_SYM);
  KVQ_BULK(KVQ_FMT_INT4_SYM, KVQ_FMT_INT4_SYM);
  KVQ_BULK(KVQ_FMT_INT4_KIVI, KVQ_FMT_INT4_KIVI);
  KVQ_BULK(KVQ_FMT_INT8_KIVI, KVQ_FMT_INT8_KIVI);
  KVQ_BULK(KVQ_FMT_INT4_KIVI, KVQ_FMT_INT8_KIVI);
  KVQ_BULK(KVQ_FMT_INT8_KIVI, KVQ_FMT_INT4_KIVI);
  KVQ_BULK(KVQ_FMT_INT8_SYM, KVQ_FMT_INT4_KIVI);
  KVQ_BULK(KVQ_FMT_INT4_KIVI, KVQ_FMT_INT8_SYM);
#undef KVQ_BULK
  if (ck == KVQ_FMT_INT4_ASYM && cv == kTileAsym) return go<KVQ_FMT_INT4_ASYM, KVQ_FMT_INT4_ASYM, 8, false, true>;
  if (ck == KVQ_FMT_INT8_SYM && cv == kTileAsym) return go<KVQ_FMT_INT8_SYM, KVQ_FMT_INT4_ASYM, 8, false, true>;
  return nullptr;
}

int64_t tiles_of(const AppendDev& d, int tok) {
  if (!d.valid) return 0;
  const int64_t lead = d.tile32 ? (d.wpos & 31) : 0;
  return (int64_t)d.B * d.H * ((lead + d.S + tok - 1) / tok);
}

}  // namespace

bool bulk_plan(const AppendDev& k, const AppendDev& v, bool local, BulkPlan& p) {
  if (!side_ok(k, p.ks) || !side_ok(v, p.vs)) return false;
  if ((k.valid ? k.S : v.S) < kBulkMinTokens) return false;
  p.ks.local = local && needs_threshold(k);
  p.vs.local = local && needs_threshold(v);
  // a missing side runs as the other one's format (its work-groups exit at once)
  p.ck = k.valid ? side_code(k) : side_code(v);
  p.cv = v.valid ? side_code(v) : side_code(k);
  // 32 tokens a wave where that gives every SIMD a few waves, fewer in shorter prompts
  const int64_t t32 = tiles_of(k, 32) > tiles_of(v, 32) ? tiles_of(k, 32) : tiles_of(v, 32);
  const bool tiled = p.ck == kTileAsym || p.cv == kTileAsym;
  p.tok = tiled || t32 >= kBulkTiles32 ? 32 : t32 >= kBulkTiles16 ? 16 : 8;
  const int64_t tiles = tiles_of(k, p.tok) > tiles_of(v, p.tok) ? tiles_of(k, p.tok) : tiles_of(v, p.tok);
  if (tiles > ((int64_t)1 << 30)) return false;
  const bool counts = (k.valid && k.st && k.status) || (v.valid && v.st && v.status);
  // (and where every work-group finds the rescue's threshold, among all rows: 4 / 8 waves, 1 x 2 heads
  // x 60 tokens in groups of 16 9.3 / 8.6 us, 1 x 4 x 250 in groups of 32 25.0 / 18.1)
  p.waves = local || (counts && tiles >= kBulkWideFrom && tiles < kBulkWideTo) ? 8 : 4;
  int64_t gx = (tiles + p.waves - 1) / p.waves;
  // at most 64 tiles a wave (its redo mask)
  const int64_t least = (tiles + 64 * p.waves - 1) / (64 * p.waves), most = kBulkWaveSlots / p.waves;
  if (gx > most) gx = most > least ? most : least;
  p.groups = (unsigned)gx;
  return pick(p.ck, p.cv, p.tok) != nullptr;
}

void append_bulk(const AppendDev& k, const AppendDev& v, const BulkPlan& p, hipStream_t st) {
  pick(p.ck, p.cv, p.tok)(k, v, p, st);
}

}  // namespace kvq

extern "C" int kvq_append_division(const float* x, const float* s, float* r, float* q, int64_t n,
                                   kvq_stream_t stream) {
  using namespace kvq;
  if (!x || !s || !r || !q || n < 0 || n > ((int64_t)1 << 31)) return fail(KVQ_ERR_INVALID, "division: bad argument");
  if (n == 0) return KVQ_OK;
  hipLaunchKernelGGL(division_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), x, s, r, q, n);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? KVQ_OK : fail(KVQ_ERR_LAUNCH, std::string("launch: ") + hipGetErrorString(e));
}
