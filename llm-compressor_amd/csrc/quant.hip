// Quantise / fake-quantise / pack kernels (bandwidth-bound: one pass, 16-byte coalesced loads).
//
// One thread owns 8 consecutive columns of a row: it loads them with one
// 16-byte access (16-bit inputs), looks the scale up once when the 8 columns
// share a group, and emits either the dequantised values, one byte per code,
// or the packed storage word (eight int4 fields in one int32, two int8 words,
// eight e4m3 bytes, or four bytes of e2m1 nibble pairs).
#include "qformat.h"

namespace {

struct QuantParams {
  const void* x;
  int x_dt;
  int64_t R, K, ldx;
  const void* scale;
  int scale_dt;
  const int8_t* zp;
  const int32_t* g_idx;
  const float* gscale;
  int fmt, bits;
  int64_t rdiv, srow, cdiv;  // scale index = (r / rdiv) * srow + (g_idx ? g_idx[c] : c / cdiv)
  int pd;                    // dtype of the quotient x / scale
  int sd;                    // dtype the dequantised value is formed in
  int out_mode;
  void* out;
  int out_dt;
  int64_t ldo;  // leading dimension of `out` in its own elements
  int64_t* shape_out;  // [2]: receives (R, K) beside the packed weight, or NULL
};

// a stored scale as fp32: the numeric dtypes, e4m3 bytes, or E8M0 exponents (2^(e-127); e = 0 is the fp32 subnormal
// 2^-127, e = 255 infinity)
__device__ __forceinline__ float load_scale(const void* p, int64_t i, int dt) {
  if (dt == LLMC_E4M3) return e4m3_decode(((const uint8_t*)p)[i]);
  if (dt == LLMC_E8M0) {
    const uint32_t e = ((const uint8_t*)p)[i];
    return __uint_as_float(e ? e << 23 : 0x00400000u);
  }
  return load_rt(p, i, dt);
}

__device__ __forceinline__ void write_shape(const QuantParams& p) {
  if (p.shape_out && blockIdx.x == 0 && threadIdx.x < 2) p.shape_out[threadIdx.x] = threadIdx.x ? p.K : p.R;
}

__device__ __forceinline__ uint32_t code_bits(float q, const QFormat& f, int bits) {
  if (f.fmt == LLMC_FMT_INT) return (uint32_t)((int)q + (1 << (bits - 1))) & ((1u << bits) - 1u);
  if (f.fmt == LLMC_FMT_FP8) return e4m3_encode(q);
  return (uint32_t)e2m1_index(fabsf(q)) | (signbit(q) ? 8u : 0u);
}

template <bool VEC>
__global__ __launch_bounds__(256) void quantize_kernel(QuantParams p) {
  const int64_t per_row = (p.K + 7) / 8;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  write_shape(p);
  if (gid >= p.R * per_row) return;
  const int64_t r = gid / per_row;
  const int64_t c0 = (gid % per_row) * 8;
  const QFormat f = make_qformat(p.fmt, p.bits);
  const float gs = p.gscale ? p.gscale[0] : 1.f;

  float xv[8];
  if (VEC && p.x_dt != LLMC_F32) {
    const uint4 v = *(const uint4*)((const uint16_t*)p.x + r * p.ldx + c0);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (p.x_dt == LLMC_BF16) {
        xv[2 * j] = __uint_as_float(w[j] << 16);
        xv[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
      } else {
        xv[2 * j] = f16_bits_to_f32((uint16_t)(w[j] & 0xffffu));
        xv[2 * j + 1] = f16_bits_to_f32((uint16_t)(w[j] >> 16));
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[j] = (c0 + j < p.K) ? load_rt(p.x, r * p.ldx + c0 + j, p.x_dt) : 0.f;
  }

  const int64_t srow_off = (r / p.rdiv) * p.srow;
  float s = 1.f, zp = 0.f;
  const bool has_zp = p.zp != nullptr;
  auto fetch = [&](int64_t c) {
    const int64_t si = srow_off + (p.g_idx ? (int64_t)p.g_idx[c] : c / p.cdiv);
    s = load_scale(p.scale, si, p.scale_dt);
    if (p.scale_dt == LLMC_E8M0) s = round_rt(s, p.sd);
    if (p.gscale) s = s / gs;  // stored scale (as fp32) / global_scale
    if (has_zp) zp = (float)p.zp[si];
  };
  if (VEC) fetch(c0);

  float qv[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (!VEC) {
      if (c0 + j >= p.K) {
        qv[j] = 0.f;
        continue;
      }
      fetch(c0 + j);
    }
    qv[j] = quantize_value(xv[j], s, zp, has_zp, p.pd, f);
    if (p.out_mode == LLMC_OUT_FAKEQUANT) qv[j] = dequantize_value(qv[j], s, zp, has_zp, p.sd);
  }

  if (p.out_mode == LLMC_OUT_FAKEQUANT) {
    if (VEC && p.out_dt != LLMC_F32) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t lo = p.out_dt == LLMC_BF16 ? f32_to_bf16_bits(qv[2 * j]) : f32_to_f16_bits(qv[2 * j]);
        const uint32_t hi = p.out_dt == LLMC_BF16 ? f32_to_bf16_bits(qv[2 * j + 1]) : f32_to_f16_bits(qv[2 * j + 1]);
        w[j] = lo | (hi << 16);
      }
      *(uint4*)((uint16_t*)p.out + r * p.ldo + c0) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (c0 + j < p.K) store_rt(p.out, r * p.ldo + c0 + j, qv[j], p.out_dt);
    }
    return;
  }

  uint32_t cb[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) cb[j] = (c0 + j < p.K) ? code_bits(qv[j], f, p.bits) : 0u;

  if (p.out_mode == LLMC_OUT_CODES) {
    // one byte per element: int8 code, e4m3 byte, or e2m1 nibble (sign in bit 3)
    uint8_t* o = (uint8_t*)p.out + r * p.ldo + c0;
    if (VEC) {
      uint32_t w0 = 0, w1 = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t b0 = f.fmt == LLMC_FMT_INT ? (uint32_t)(uint8_t)(int8_t)(int)qv[j] : cb[j];
        const uint32_t b1 = f.fmt == LLMC_FMT_INT ? (uint32_t)(uint8_t)(int8_t)(int)qv[j + 4] : cb[j + 4];
        w0 |= b0 << (8 * j);
        w1 |= b1 << (8 * j);
      }
      *(uint2*)o = make_uint2(w0, w1);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (c0 + j < p.K) o[j] = f.fmt == LLMC_FMT_INT ? (uint8_t)(int8_t)(int)qv[j] : (uint8_t)cb[j];
    }
    return;
  }

  // LLMC_OUT_PACKED
  if (f.fmt == LLMC_FMT_FP4) {
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) w |= cb[j] << (4 * j);  // even column in the low nibble of each byte
    uint8_t* o = (uint8_t*)p.out + r * p.ldo + c0 / 2;
    if (VEC) {
      *(uint32_t*)o = w;
    } else {
      for (int j = 0; j < 4; ++j)
        if (c0 + 2 * j < p.K) o[j] = (uint8_t)(w >> (8 * j));
    }
  } else if (f.fmt == LLMC_FMT_FP8) {
    uint8_t* o = (uint8_t*)p.out + r * p.ldo + c0;
    for (int j = 0; j < 8; ++j)
      if (c0 + j < p.K) o[j] = (uint8_t)cb[j];
  } else {
    // offset-binary fields, element j of a word at bit j*bits, 32/bits elements per int32 word
    const int pf = 32 / p.bits;
    uint32_t* o = (uint32_t*)p.out + r * p.ldo;
    if (pf == 8) {
      uint32_t w = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) w |= cb[j] << (4 * j);
      o[c0 / 8] = w;
    } else if (pf == 4) {
      uint32_t w0 = 0, w1 = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w0 |= cb[j] << (8 * j);
        w1 |= cb[j + 4] << (8 * j);
      }
      o[c0 / 4] = w0;
      if (c0 + 4 < p.K) o[c0 / 4 + 1] = w1;
    } else {
      // other widths (pf = 16, 10, 6, 5): a word may straddle this thread's 8 columns
      for (int j = 0; j < 8; ++j)
        if (c0 + j < p.K) atomicOr(&o[(c0 + j) / pf], cb[j] << (((c0 + j) % pf) * p.bits));
    }
  }
}

// ---- the common case: 16-bit input with K % 8 == 0, scales in the input's dtype, fp32 or stored codes,
// power-of-two (or whole-row) column groups, no g_idx, 4/8-bit ints, e4m3 or e2m1.
// A lane owns E consecutive columns (16; 8 where K is not a multiple of 16) and everything the format decides is a
// template parameter, so the per-element path is branch-free: shared-divisor division, rounding to the quotient's
// dtype, clamp, and the hardware e4m3/e2m1 conversions.  The lanes are numbered over the whole matrix, not per
// row: with a workgroup per row, 256 columns kept 16 of its 256 lanes busy and a 1664-column row 104 of them.
template <int XDT>
__device__ __forceinline__ void unpack8(const uint4& v, float* x) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (XDT == LLMC_BF16) {
      x[2 * j] = __uint_as_float(w[j] << 16);
      x[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    } else {
      x[2 * j] = f16_bits_to_f32((uint16_t)(w[j] & 0xffffu));
      x[2 * j + 1] = f16_bits_to_f32((uint16_t)(w[j] >> 16));
    }
  }
}

// N consecutive 32-bit words as one store
template <int N>
__device__ __forceinline__ void store_words(void* dst, const uint32_t (&w)[N]) {
  if constexpr (N == 4)
    *(uint4*)dst = make_uint4(w[0], w[1], w[2], w[3]);
  else if constexpr (N == 2)
    *(uint2*)dst = make_uint2(w[0], w[1]);
  else
    *(uint32_t*)dst = w[0];
}

// How the rows of a launch are walked.  `row_mul` is floor(2^64 / units per row) + 1 (0 = one unit per row): the high
// word of its product with a unit number below 2^32 is the row number.
struct RowsWalk {
  uint32_t units, per_row;
  uint64_t row_mul;
  int cshift;  // log2 of the columns per scale (31: one scale per row)
  int rshift;  // log2 of the rows per scale (63: one for all rows)
  int lanes;   // SM >= SM_OWN: lanes that share a group
  uint32_t turned;  // the first `turned` blocks (a multiple of eight) take the last rows first
};

// Whoever produced or observed the input went through it from the front, so that what of a large one the memory-side cache
// (256 MB) still holds is its end: the last rows come first then, eight blocks at a time, so that a block stays on its XCD,
// whose L2 may hold its part.  In us, in order / turned: after an observer, W4A16 14336 x 4096 22.7 / 22.0, 28672 x 8192 94 / 89,
// 128256 x 4096 218 / 211, FP8 28672 x 8192 108 / 105; MXFP4 of activations just written, 8192 x 14336 84 / 81.5, 2048 x 14336
// (59 MB) 19.6 / 19.5.  Below that the order only costs: 2048 x 4096 8.0 / 8.4, W4A16 1024 x 4096 4.1 / 4.4 (9.3 and 5.3 block by
// block, which gives every block to another XCD).
constexpr int64_t TURN_MIN_BYTES = 64 << 20;

// where the scale of a lane's columns comes from
enum {
  SM_SAME = 0,      // stored in the input's 16-bit dtype
  SM_F32 = 1,       // stored in fp32 (or as e4m3 without a global scale)
  SM_GLOBAL = 2,    // stored scale / global scale, in fp32
  SM_E8M0 = 3,      // stored as E8M0 exponents
  SM_OWN = 4,       // dynamic: from the group's own largest magnitude, in the input's dtype
  SM_OWN_MX = 5,    // dynamic, E8M0
  SM_OWN_NVFP4 = 6  // dynamic, e4m3 under the global scale
};

// Dynamic groups (SM_OWN*): the group's lanes are neighbours, so its largest magnitude is a few xor-shuffles away and
// the value is quantised in the pass that observed it.  As min-max, qparams and quantise kernels this read the
// activation twice and cost three launches: [1084 x 3168] bf16 with MXFP4 groups took 92 us, most of it host.
template <int XDT, int SM, int FMT, bool HAS_ZP, int OUT, int E>
__global__ __launch_bounds__(256) void quantize_rows_kernel(QuantParams p, RowsWalk walk) {
  constexpr bool S32 = SM == SM_F32 || SM == SM_GLOBAL || SM == SM_OWN_NVFP4;
  constexpr int PD = S32 ? LLMC_F32 : XDT;  // dtype of the quotient and of the dequantised value
  write_shape(p);
  const uint32_t b = blockIdx.x;
  const uint32_t unit = (b < walk.turned ? walk.turned - 8u - (b & ~7u) + (b & 7u) : b) * 256u + threadIdx.x;
  if (unit >= walk.units) return;
  const uint32_t row = walk.row_mul ? (uint32_t)__umul64hi((uint64_t)unit, walk.row_mul) : unit;
  const int64_t r = row;
  const int c0 = (int)(unit - row * walk.per_row) * E;
  const uint16_t* xr = (const uint16_t*)p.x + r * p.ldx;
  const QFormat f = make_qformat(FMT, p.bits);
  float gs = 1.f;
  if (SM == SM_GLOBAL || SM == SM_OWN_NVFP4) gs = p.gscale[0];

  {
    uint4 raw[E / 8];
#pragma unroll
    for (int k = 0; k < E / 8; ++k) raw[k] = *(const uint4*)(xr + c0 + 8 * k);
    const int64_t si = (r >> walk.rshift) * p.srow + (c0 >> walk.cshift);
    float s;
    if (SM == SM_SAME)
      s = load_as_f32<XDT>(p.scale, si);
    else if (SM == SM_F32)
      s = p.scale_dt == LLMC_E4M3 ? load_scale(p.scale, si, LLMC_E4M3) : ((const float*)p.scale)[si];
    else if (SM == SM_GLOBAL)
      s = load_scale(p.scale, si, p.scale_dt) / gs;
    else if (SM == SM_E8M0)
      s = round_to<XDT>(load_scale(p.scale, si, LLMC_E8M0));
    else
      s = 0.f;
    const float zp = HAS_ZP ? (float)p.zp[si] : 0.f;
    float x[E], v[E];
#pragma unroll
    for (int k = 0; k < E / 8; ++k) unpack8<XDT>(raw[k], x + 8 * k);
    if (SM >= SM_OWN) {
      float amax = 0.f;
#pragma unroll
      for (int j = 0; j < E; ++j) amax = fmaxf(amax, fabsf(x[j]));
      for (int o = walk.lanes >> 1; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
      constexpr int mode = SM == SM_OWN_MX ? LLMC_SCALE_MXFP4 : SM == SM_OWN_NVFP4 ? LLMC_SCALE_NVFP4 : LLMC_SCALE_PLAIN;
      float zero;
      int e;
      qparams_from_minmax(-amax, amax, XDT, f, true, mode, gs, &s, &zero, &e);
      if (SM == SM_OWN_MX) s = __uint_as_float(e ? (uint32_t)e << 23 : 0x00400000u);
      if (SM == SM_OWN_NVFP4) s = s / gs;
    }
    const FastDiv d = make_fastdiv(s);
    bool redo;
    if (XDT == LLMC_BF16 && !S32) {
      // bf16 values over a bf16 scale: the rounded quotient is one multiply away (see qformat.h)
      Bf16Range rg = bf16_range_init();
#pragma unroll
      for (int k = 0; k < E / 8; ++k) {
        bf16_range_add(rg, raw[k].x); bf16_range_add(rg, raw[k].y); bf16_range_add(rg, raw[k].z); bf16_range_add(rg, raw[k].w);
      }
      redo = !(bf16_inputs_plain(rg) & bf16_scale_plain(s));
#pragma unroll
      for (int j = 0; j < E; ++j) v[j] = x[j] * d.y;
    } else {
      bool big = false, small = false;
#pragma unroll
      for (int j = 0; j < E; ++j) {
        v[j] = fastdiv(x[j], d);
        big = big | !fastdiv_big_ok(v[j]);
        small = small | fastdiv_small(v[j]);
      }
      redo = big | !d.ok;
      if (small) {
#pragma unroll
        for (int j = 0; j < E; ++j) redo = redo | (fastdiv_small(v[j]) & (x[j] != 0.f));
      }
    }
    if (redo) {
      // out-of-range divisor or quotient, NaN: the plain division, then the same tail
#pragma unroll
      for (int j = 0; j < E; ++j) {
        v[j] = round_rt(x[j] / s, PD);
        v[j] = HAS_ZP ? round_rt(v[j] + zp, PD) : v[j] + 0.0f;
        v[j] = fminf(fmaxf(v[j], f.qmin), f.qmax);
      }
    } else {
#pragma unroll
      for (int j = 0; j < E; ++j) {
        if (!S32) v[j] = round16_finite<XDT>(v[j]);
        if (HAS_ZP)
          v[j] = S32 ? v[j] + zp : round16_finite<XDT>(v[j] + zp);
        else if (FMT != LLMC_FMT_INT || OUT == LLMC_OUT_FAKEQUANT)
          v[j] = v[j] + 0.0f;  // the reference adds a zero zero-point: -0.0 becomes +0.0
        v[j] = __builtin_amdgcn_fmed3f(v[j], f.qmin, f.qmax);
      }
    }

    // element codes: e4m3 bytes / e2m1 nibbles via the conversion instructions
    uint32_t fp8w[E / 4] = {}, fp4w[E / 8] = {};
    if (FMT == LLMC_FMT_FP8) {
#pragma unroll
      for (int j = 0; j < E / 2; ++j) fp8w[j >> 1] |= hw_e4m3_pair(v[2 * j], v[2 * j + 1]) << (16 * (j & 1));
    } else if (FMT == LLMC_FMT_FP4) {
#pragma unroll
      for (int j = 0; j < E / 2; ++j) fp4w[j >> 2] |= hw_e2m1_pair(v[2 * j], v[2 * j + 1]) << (8 * (j & 3));
    }

    if (OUT == LLMC_OUT_FAKEQUANT) {
      if (FMT == LLMC_FMT_INT) {
#pragma unroll
        for (int j = 0; j < E; ++j) v[j] = rintf(v[j]);
      } else if (FMT == LLMC_FMT_FP8) {
#pragma unroll
        for (int j = 0; j < E / 2; ++j) {
          const f32x2_t t = hw_e4m3_pair_decode(fp8w[j >> 1] >> (16 * (j & 1)));
          v[2 * j] = t.x;
          v[2 * j + 1] = t.y;
        }
      } else {
#pragma unroll
        for (int j = 0; j < E / 2; ++j) {
          const f32x2_t t = hw_e2m1_pair_decode(fp4w[j >> 2] >> (8 * (j & 3)));
          v[2 * j] = t.x;
          v[2 * j + 1] = t.y;
        }
      }
#pragma unroll
      for (int j = 0; j < E; ++j) {
        if (HAS_ZP) v[j] = round_rt(v[j] - zp, PD);
        v[j] *= s;  // rounding to PD, then to the output's dtype, is one rounding
      }
      uint16_t* o = (uint16_t*)p.out + r * p.ldo + c0;
#pragma unroll
      for (int k = 0; k < E / 8; ++k)
        *(uint4*)(o + 8 * k) = make_uint4(pack16<XDT>(v[8 * k], v[8 * k + 1]), pack16<XDT>(v[8 * k + 2], v[8 * k + 3]),
                                          pack16<XDT>(v[8 * k + 4], v[8 * k + 5]), pack16<XDT>(v[8 * k + 6], v[8 * k + 7]));
      return;
    }

    if (FMT == LLMC_FMT_FP8) {  // bytes either way
      store_words<E / 4>((uint8_t*)p.out + r * p.ldo + c0, fp8w);
    } else if (FMT == LLMC_FMT_FP4) {
      if (OUT == LLMC_OUT_PACKED) {
        store_words<E / 8>((uint8_t*)p.out + r * p.ldo + (c0 >> 1), fp4w);
      } else {  // one nibble per byte
        uint32_t w[E / 4];
#pragma unroll
        for (int k = 0; k < E / 4; ++k) {
          const uint32_t h = (fp4w[k >> 1] >> (16 * (k & 1))) & 0xffffu;
          w[k] = (h & 0xfu) | ((h & 0xf0u) << 4) | ((h & 0xf00u) << 8) | ((h & 0xf000u) << 12);
        }
        store_words<E / 4>((uint8_t*)p.out + r * p.ldo + c0, w);
      }
    } else {
      // v + 1.5*2^23 rounds v to the nearest-even integer and leaves it, two's complement, in the
      // low mantissa bits; funnel shifts collect the low 4 or 8 bits of each element
      uint32_t q[E];
#pragma unroll
      for (int j = 0; j < E; ++j) q[j] = __float_as_uint(v[j] + 12582912.0f);
      if (OUT == LLMC_OUT_CODES || p.bits == 8) {
        // int8 codes, or int8 fields (offset binary) four to a word: the same byte positions
        uint32_t w[E / 4] = {};
        const uint32_t flip = OUT == LLMC_OUT_CODES ? 0u : 0x80808080u;
#pragma unroll
        for (int j = 0; j < E; ++j) w[j >> 2] = __builtin_amdgcn_alignbit(q[j], w[j >> 2], 8);
#pragma unroll
        for (int k = 0; k < E / 4; ++k) w[k] ^= flip;
        if (OUT == LLMC_OUT_CODES)
          store_words<E / 4>((uint8_t*)p.out + r * p.ldo + c0, w);
        else
          store_words<E / 4>((uint32_t*)p.out + r * p.ldo + (c0 >> 2), w);
      } else {  // 4-bit fields, offset binary
        uint32_t w[E / 8] = {};
#pragma unroll
        for (int j = 0; j < E; ++j) w[j >> 3] = __builtin_amdgcn_alignbit(q[j], w[j >> 3], 4);
#pragma unroll
        for (int k = 0; k < E / 8; ++k) w[k] ^= 0x88888888u;
        store_words<E / 8>((uint32_t*)p.out + r * p.ldo + (c0 >> 3), w);
      }
    }
  }
}

template <int XDT, int SM, int FMT, bool HAS_ZP, int OUT>
void launch_rows_e(const QuantParams& p, const RowsWalk& w, int e, hipStream_t st) {
  const dim3 grid((w.units + 255) / 256), block(256);
  // 8 columns per lane only for scales that a row, a column block or the matrix shares: the others come in groups
  // of 16 or more, so K is a multiple of 16 there
  if constexpr (SM == SM_SAME || SM == SM_F32) {
    if (e == 8) {
      hipLaunchKernelGGL((quantize_rows_kernel<XDT, SM, FMT, HAS_ZP, OUT, 8>), grid, block, 0, st, p, w);
      return;
    }
  }
  hipLaunchKernelGGL((quantize_rows_kernel<XDT, SM, FMT, HAS_ZP, OUT, 16>), grid, block, 0, st, p, w);
}

template <int XDT, int SM, int FMT, bool HAS_ZP>
void launch_rows_out(const QuantParams& p, const RowsWalk& w, int e, hipStream_t st) {
  if (SM >= SM_OWN || p.out_mode == LLMC_OUT_FAKEQUANT)
    launch_rows_e<XDT, SM, FMT, HAS_ZP, LLMC_OUT_FAKEQUANT>(p, w, e, st);
  else if constexpr (SM < SM_OWN) {
    if (p.out_mode == LLMC_OUT_CODES)
      launch_rows_e<XDT, SM, FMT, HAS_ZP, LLMC_OUT_CODES>(p, w, e, st);
    else
      launch_rows_e<XDT, SM, FMT, HAS_ZP, LLMC_OUT_PACKED>(p, w, e, st);
  }
}

template <int XDT, int SM>
void launch_rows_fmt(const QuantParams& p, const RowsWalk& w, int e, hipStream_t st) {
  if constexpr (SM == SM_E8M0 || SM == SM_OWN_MX || SM == SM_OWN_NVFP4) {  // fp4 formats only
    launch_rows_out<XDT, SM, LLMC_FMT_FP4, false>(p, w, e, st);
  } else if (p.fmt == LLMC_FMT_INT) {
    if constexpr (SM < SM_OWN) {
      if (p.zp) {
        launch_rows_out<XDT, SM, LLMC_FMT_INT, true>(p, w, e, st);
        return;
      }
    }
    launch_rows_out<XDT, SM, LLMC_FMT_INT, false>(p, w, e, st);
  } else if (p.fmt == LLMC_FMT_FP8) {
    launch_rows_out<XDT, SM, LLMC_FMT_FP8, false>(p, w, e, st);
  } else {
    launch_rows_out<XDT, SM, LLMC_FMT_FP4, false>(p, w, e, st);
  }
}

template <int XDT>
void launch_rows_sm(int sm, const QuantParams& p, const RowsWalk& w, int e, hipStream_t st) {
  switch (sm) {
    case SM_SAME: launch_rows_fmt<XDT, SM_SAME>(p, w, e, st); break;
    case SM_F32: launch_rows_fmt<XDT, SM_F32>(p, w, e, st); break;
    case SM_GLOBAL: launch_rows_fmt<XDT, SM_GLOBAL>(p, w, e, st); break;
    case SM_E8M0: launch_rows_fmt<XDT, SM_E8M0>(p, w, e, st); break;
    case SM_OWN: launch_rows_fmt<XDT, SM_OWN>(p, w, e, st); break;
    case SM_OWN_MX:  // the exponent is read off bf16 values
      if constexpr (XDT == LLMC_BF16) launch_rows_fmt<XDT, SM_OWN_MX>(p, w, e, st);
      break;
    default: launch_rows_fmt<XDT, SM_OWN_NVFP4>(p, w, e, st);
  }
}

int log2_exact(int64_t v) {  // log2 of a power of two, -1 otherwise
  if (v <= 0 || (v & (v - 1))) return -1;
  int n = 0;
  while ((1LL << n) < v) ++n;
  return n;
}

// units are numbered in 32 bits, with room for the last workgroup's lanes past the end
bool units_fit(int64_t R, int64_t per_row) { return R <= ((1LL << 32) - 256) / per_row; }

void walk_rows(RowsWalk& w, int64_t R, int64_t K, int e) {
  w.per_row = (uint32_t)(K / e);
  w.units = (uint32_t)(R * w.per_row);
  w.row_mul = w.per_row > 1 ? ~0ull / w.per_row + 1 : 0;
  w.lanes = 1;
  w.turned = R * K * 2 > TURN_MIN_BYTES ? (w.units + 255) / 256 & ~7u : 0u;
}

// launches the row kernel when the call fits its assumptions; false = use the general kernel
bool try_launch_rows(const QuantParams& p, hipStream_t st) {
  if (p.x_dt == LLMC_F32 || p.g_idx || p.K % 8 || p.ldx % 8 || ((uintptr_t)p.x & 15)) return false;
  const int e = p.K % 16 ? 8 : 16;
  if (p.K > (1LL << 30) || !units_fit(p.R, p.K / e)) return false;
  const int sm = p.gscale ? SM_GLOBAL
                 : p.scale_dt == LLMC_E8M0 ? SM_E8M0
                 : p.scale_dt == LLMC_F32 || p.scale_dt == LLMC_E4M3 ? SM_F32 : SM_SAME;
  if (sm == SM_SAME && p.scale_dt != p.x_dt) return false;
  if (p.scale_dt == LLMC_E8M0 && (p.gscale || p.fmt != LLMC_FMT_FP4)) return false;
  if (e == 8 && sm != SM_SAME && sm != SM_F32) return false;
  if (p.zp && p.fmt != LLMC_FMT_INT) return false;
  if (p.fmt == LLMC_FMT_INT && p.bits != 4 && p.bits != 8) return false;
  RowsWalk w;
  walk_rows(w, p.R, p.K, e);
  w.cshift = p.cdiv >= p.K ? 31 : log2_exact(p.cdiv);
  w.rshift = p.rdiv >= p.R ? 63 : log2_exact(p.rdiv);
  if (w.cshift < 0 || w.rshift < 0 || (1LL << w.cshift) < e) return false;
  // a lane's output, as one store
  const int64_t ldo_bytes = p.ldo * (p.out_mode == LLMC_OUT_FAKEQUANT ? 2 : p.out_mode == LLMC_OUT_PACKED && p.fmt == LLMC_FMT_INT ? 4 : 1);
  int store;
  if (p.out_mode == LLMC_OUT_FAKEQUANT) {
    if (p.out_dt != p.x_dt) return false;
    store = 16;
  } else if (p.out_mode == LLMC_OUT_CODES || p.fmt == LLMC_FMT_FP8 || (p.fmt == LLMC_FMT_INT && p.bits == 8)) {
    store = e;
  } else {
    store = e / 2;
  }
  if (ldo_bytes % store || ((uintptr_t)p.out & (store - 1))) return false;
  if (p.x_dt == LLMC_BF16)
    launch_rows_sm<LLMC_BF16>(sm, p, w, e, st);
  else
    launch_rows_sm<LLMC_F16>(sm, p, w, e, st);
  return true;
}

// Per-token dynamic quantisation of rows that are not whole 16-byte chunks: one workgroup per row.  The row is staged
// in LDS while its absmax is reduced, so HBM sees one read and one write per element.
template <int DT>
__global__ __launch_bounds__(256) void dynamic_token_kernel(const void* __restrict__ x, int64_t ldx, int K,
                                                            int fmt, int bits, int out_mode,
                                                            void* __restrict__ out, int64_t ldo,
                                                            void* __restrict__ scale_out) {
  extern __shared__ __attribute__((aligned(16))) uint16_t row[];
  __shared__ float wred[4];
  const int64_t r = blockIdx.x;
  const uint16_t* xr = (const uint16_t*)x + r * ldx;
  const bool vec = (K % 8 == 0) && (ldx % 8 == 0) && (((uintptr_t)x & 15) == 0);
  float amax = 0.f;
  if (vec) {
    for (int c = threadIdx.x * 8; c < K; c += 256 * 8) {
      const uint4 v = *(const uint4*)(xr + c);
      *(uint4*)(row + c) = v;
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float lo = load_as_f32<DT>(&w[j], 0), hi = load_as_f32<DT>(&w[j], 1);
        amax = fmaxf(amax, fmaxf(fabsf(lo), fabsf(hi)));
      }
    }
  } else {
    for (int c = threadIdx.x; c < K; c += 256) {
      row[c] = xr[c];
      amax = fmaxf(amax, fabsf(load_as_f32<DT>(xr, c)));
    }
  }
  amax = wave_max(amax);
  if ((threadIdx.x & 63) == 0) wred[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wred[0], wred[1]), fmaxf(wred[2], wred[3]));
  const QFormat f = make_qformat(fmt, bits);
  float s = round_to<DT>(amax / ((f.qmax - f.qmin) * 0.5f));
  if (s == 0.f) s = dtype_eps(DT);
  if (threadIdx.x == 0 && scale_out) store_from_f32<DT>(scale_out, r, s);
  for (int c = threadIdx.x * 8; c < K; c += 256 * 8) {
    float q[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float xv = (c + j < K) ? load_as_f32<DT>(row, c + j) : 0.f;
      q[j] = quantize_value(xv, s, 0.f, false, DT, f);
    }
    if (out_mode == LLMC_OUT_FAKEQUANT) {
      uint16_t o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = dequantize_value(q[j], s, 0.f, false, DT);
        o[j] = DT == LLMC_BF16 ? f32_to_bf16_bits(d) : f32_to_f16_bits(d);
      }
      uint16_t* orow = (uint16_t*)out + r * ldo;
      if (vec && (ldo % 8 == 0) && (((uintptr_t)out & 15) == 0)) {
        *(uint4*)(orow + c) = make_uint4(o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16),
                                         o[4] | ((uint32_t)o[5] << 16), o[6] | ((uint32_t)o[7] << 16));
      } else {
        for (int j = 0; j < 8; ++j)
          if (c + j < K) orow[c + j] = o[j];
      }
    } else {
      uint8_t* orow = (uint8_t*)out + r * ldo;
      uint32_t w0 = 0, w1 = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w0 |= code_bits(q[j], f, bits) << (8 * j);
        w1 |= code_bits(q[j + 4], f, bits) << (8 * j);
      }
      if (f.fmt == LLMC_FMT_INT) {
        w0 = w1 = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w0 |= (uint32_t)(uint8_t)(int8_t)(int)q[j] << (8 * j);
          w1 |= (uint32_t)(uint8_t)(int8_t)(int)q[j + 4] << (8 * j);
        }
      }
      if (vec && (ldo % 8 == 0) && (((uintptr_t)out & 7) == 0)) {
        *(uint2*)(orow + c) = make_uint2(w0, w1);
      } else {
        for (int j = 0; j < 8; ++j)
          if (c + j < K) orow[c + j] = (uint8_t)((j < 4 ? w0 : w1) >> (8 * (j & 3)));
      }
    }
  }
}

// Per-token dynamic quantisation of rows of whole 16-byte chunks, held in registers between the absmax reduction and the
// quantisation (one HBM read, one write).  WAVES wavefronts share a row: one up to 8192 elements (no LDS, no
// barrier, four rows per workgroup), 4 up to 16384, 16 beyond.  Chunk i of lane l is 64 * WAVES * i + l.
// 8192 x 14336 bf16: 166 us through the LDS-staged kernel above (plain divisions and a re-read of the row from LDS).
template <int DT, int NC, int FMT, int OUT, int WAVES>
__global__ __launch_bounds__(WAVES == 16 ? 1024 : 256) void dynamic_token_wave_kernel(
    const void* __restrict__ x, int64_t ldx, int64_t N, int K, int bits, void* __restrict__ out, int64_t ldo,
    void* __restrict__ scale_out) {
  constexpr int LANES = 64 * WAVES;
  const int lane = WAVES == 1 ? threadIdx.x & 63 : threadIdx.x;
  const int64_t r = WAVES == 1 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  if (r >= N) return;
  const uint16_t* xr = (const uint16_t*)x + r * ldx;
  const int nchunk = K >> 3;
  uint4 raw[NC];
  u16x2_t m = {0, 0};  // packed max of 15-bit magnitudes (magnitude bits order like the values)
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = i * LANES + lane;
    raw[i] = c < nchunk ? *(const uint4*)(xr + (c << 3)) : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t a = w[j] & 0x7fff7fffu;
      u16x2_t av;
      __builtin_memcpy(&av, &a, 4);
      m = __builtin_elementwise_max(m, av);
    }
  }
  uint32_t mm = max((uint32_t)m.x, (uint32_t)m.y);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mm = max(mm, (uint32_t)__shfl_xor((int)mm, o, 64));
  if constexpr (WAVES > 1) {
    __shared__ uint32_t wave_mm[WAVES];
    if ((threadIdx.x & 63) == 0) wave_mm[threadIdx.x >> 6] = mm;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mm = max(mm, wave_mm[w]);
  }
  const float amax = DT == LLMC_BF16 ? bf16_bits_to_f32((uint16_t)mm) : f16_bits_to_f32((uint16_t)mm);
  const QFormat f = make_qformat(FMT, bits);
  float s = round_to<DT>(amax / ((f.qmax - f.qmin) * 0.5f));
  if (s == 0.f) s = dtype_eps(DT);
  if (lane == 0 && scale_out) store_from_f32<DT>(scale_out, r, s);
  const FastDiv d = make_fastdiv(s);
  // bf16 rows: the scale is a bf16 value too, so the rounded quotient is one multiply away (see qformat.h);
  // the row's largest magnitude is known, only values far below it need the guard
  const bool plain_scale = DT == LLMC_BF16 && bf16_scale_plain(s) && mm < ((127u + 96u) << 7);

#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int c = i * LANES + lane;
    if (c >= nchunk) break;
    float xv[8], v[8];
    unpack8<DT>(raw[i], xv);
    bool redo;
    if (DT == LLMC_BF16) {
      Bf16Range rg = bf16_range_init();
      bf16_range_add(rg, raw[i].x); bf16_range_add(rg, raw[i].y); bf16_range_add(rg, raw[i].z); bf16_range_add(rg, raw[i].w);
      redo = !(bf16_inputs_plain(rg) & plain_scale);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = xv[j] * d.y;
    } else {
      bool big = false, small = false;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[j] = fastdiv(xv[j], d);
        big = big | !fastdiv_big_ok(v[j]);
        small = small | fastdiv_small(v[j]);
      }
      redo = big | !d.ok;
      if (small) {
#pragma unroll
        for (int j = 0; j < 8; ++j) redo = redo | (fastdiv_small(v[j]) & (xv[j] != 0.f));
      }
    }
    if (redo) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = fminf(fmaxf(round_to<DT>(xv[j] / s) + 0.0f, f.qmin), f.qmax);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = __builtin_amdgcn_fmed3f(round16_finite<DT>(v[j]) + 0.0f, f.qmin, f.qmax);
    }
    uint32_t cw[2] = {0u, 0u};  // the eight element bytes
    if (FMT == LLMC_FMT_FP8) {
#pragma unroll
      for (int j = 0; j < 4; ++j) cw[j >> 1] |= hw_e4m3_pair(v[2 * j], v[2 * j + 1]) << (16 * (j & 1));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        cw[j >> 2] = __builtin_amdgcn_alignbit(__float_as_uint(v[j] + 12582912.0f), cw[j >> 2], 8);
    }
    if (OUT == LLMC_OUT_CODES) {
      *(uint2*)((uint8_t*)out + r * ldo + (c << 3)) = make_uint2(cw[0], cw[1]);
    } else {
      if (FMT == LLMC_FMT_FP8) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x2_t t = hw_e4m3_pair_decode(cw[j >> 1] >> (16 * (j & 1)));
          v[2 * j] = t.x;
          v[2 * j + 1] = t.y;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = rintf(v[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] *= s;
      *(uint4*)((uint16_t*)out + r * ldo + (c << 3)) =
          make_uint4(pack16<DT>(v[0], v[1]), pack16<DT>(v[2], v[3]), pack16<DT>(v[4], v[5]), pack16<DT>(v[6], v[7]));
    }
  }
}

template <int DT, int NC, int WAVES>
void launch_token_wave(const void* x, int64_t ldx, int64_t N, int K, int fmt, int bits, int out_mode, void* out,
                       int64_t ldo, void* scale_out, hipStream_t st) {
  const dim3 grid((unsigned)(WAVES == 1 ? (N + 3) / 4 : N)), block(WAVES == 16 ? 1024 : 256);
#define LLMC_TOK(F, O)                                                                                              \
  hipLaunchKernelGGL((dynamic_token_wave_kernel<DT, NC, F, O, WAVES>), grid, block, 0, st, x, ldx, N, K, bits, out, \
                     ldo, scale_out)
  if (fmt == LLMC_FMT_FP8) {
    if (out_mode == LLMC_OUT_CODES) LLMC_TOK(LLMC_FMT_FP8, LLMC_OUT_CODES);
    else LLMC_TOK(LLMC_FMT_FP8, LLMC_OUT_FAKEQUANT);
  } else {
    if (out_mode == LLMC_OUT_CODES) LLMC_TOK(LLMC_FMT_INT, LLMC_OUT_CODES);
    else LLMC_TOK(LLMC_FMT_INT, LLMC_OUT_FAKEQUANT);
  }
#undef LLMC_TOK
}

// A row takes one wavefront while its chunks fit that wavefront's registers and there are rows enough for every SIMD
// (1024 of them); fewer or longer rows are shared by four, which also shortens a decode step's single row.
template <int DT>
void launch_token_wave_nc(const void* x, int64_t ldx, int64_t N, int K, int fmt, int bits, int out_mode,
                          void* out, int64_t ldo, void* scale_out, hipStream_t st) {
  const int chunks = K / 8;
  if (chunks > 2048) launch_token_wave<DT, 8, 16>(x, ldx, N, K, fmt, bits, out_mode, out, ldo, scale_out, st);
  else if (chunks > 1024) launch_token_wave<DT, 8, 4>(x, ldx, N, K, fmt, bits, out_mode, out, ldo, scale_out, st);
  else if (chunks > 128 && N < 1024)
    launch_token_wave<DT, 4, 4>(x, ldx, N, K, fmt, bits, out_mode, out, ldo, scale_out, st);
  else if (chunks <= 128) launch_token_wave<DT, 2, 1>(x, ldx, N, K, fmt, bits, out_mode, out, ldo, scale_out, st);
  else if (chunks <= 512) launch_token_wave<DT, 8, 1>(x, ldx, N, K, fmt, bits, out_mode, out, ldo, scale_out, st);
  else launch_token_wave<DT, 16, 1>(x, ldx, N, K, fmt, bits, out_mode, out, ldo, scale_out, st);
}

__global__ void fill_u32_kernel(uint32_t* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

int promote(int a, int b) {
  if (a == LLMC_F32 || b == LLMC_F32) return LLMC_F32;
  return a == b ? a : LLMC_F32;
}

}  // namespace

extern "C" int llmc_quantize(const void* x, int32_t x_dtype, int64_t R, int64_t K, int64_t ldx,
                             const void* scale, int32_t scale_dtype, const int8_t* zero_point,
                             const int32_t* g_idx, const float* global_scale, int32_t fmt, int32_t num_bits,
                             int64_t row_div, int64_t scale_row_stride, int64_t col_div, int32_t out_mode,
                             void* out, int32_t out_dtype, int64_t ldo, void* stream) {
  return llmc_quantize_shaped(x, x_dtype, R, K, ldx, scale, scale_dtype, zero_point, g_idx, global_scale, fmt, num_bits,
                              row_div, scale_row_stride, col_div, out_mode, out, out_dtype, ldo, nullptr, stream);
}

extern "C" int llmc_quantize_shaped(const void* x, int32_t x_dtype, int64_t R, int64_t K, int64_t ldx,
                                    const void* scale, int32_t scale_dtype, const int8_t* zero_point,
                                    const int32_t* g_idx, const float* global_scale, int32_t fmt, int32_t num_bits,
                                    int64_t row_div, int64_t scale_row_stride, int64_t col_div, int32_t out_mode,
                                    void* out, int32_t out_dtype, int64_t ldo, int64_t* shape_out, void* stream) {
  LLMC_CHECK_ARG(x && R > 0 && K > 0, 1);
  LLMC_CHECK_ARG(x_dtype >= 0 && x_dtype <= 2, 2);
  LLMC_CHECK_ARG(ldx >= K, 5);
  LLMC_CHECK_ARG(scale, 6);
  LLMC_CHECK_ARG(scale_dtype >= 0 && scale_dtype <= LLMC_E8M0, 7);
  LLMC_CHECK_ARG(fmt >= 0 && fmt <= 2, 11);
  LLMC_CHECK_ARG(fmt != LLMC_FMT_INT || (num_bits >= 2 && num_bits <= 8), 12);
  LLMC_CHECK_ARG(row_div > 0 && col_div > 0 && scale_row_stride >= 0, 13);
  LLMC_CHECK_ARG(out_mode >= 0 && out_mode <= 2, 16);
  LLMC_CHECK_ARG(out, 17);
  hipStream_t st = (hipStream_t)stream;
  QuantParams p;
  p.x = x; p.x_dt = x_dtype; p.R = R; p.K = K; p.ldx = ldx;
  p.scale = scale; p.scale_dt = scale_dtype; p.zp = zero_point; p.g_idx = g_idx; p.gscale = global_scale;
  p.fmt = fmt; p.bits = fmt == LLMC_FMT_INT ? num_bits : (fmt == LLMC_FMT_FP8 ? 8 : 4);
  p.rdiv = row_div; p.srow = scale_row_stride; p.cdiv = col_div;
  // stored codes stand for fp32 values (e4m3) or for powers of two in the input's 16-bit dtype (E8M0)
  const int eff_scale_dt = global_scale || scale_dtype == LLMC_E4M3 ? LLMC_F32
                           : scale_dtype == LLMC_E8M0 ? (x_dtype == LLMC_F32 ? LLMC_BF16 : x_dtype) : scale_dtype;
  p.pd = promote(x_dtype, eff_scale_dt);
  p.sd = eff_scale_dt;
  p.out_mode = out_mode; p.out = out; p.out_dt = out_dtype; p.ldo = ldo; p.shape_out = shape_out;

  if (try_launch_rows(p, st)) {
    LLMC_LAUNCH_STATUS();
    return 0;
  }
  bool vec = (K % 8 == 0) && (col_div % 8 == 0) && g_idx == nullptr && (((uintptr_t)x & 15) == 0) &&
             (x_dtype == LLMC_F32 || ldx % 8 == 0);
  if (out_mode == LLMC_OUT_FAKEQUANT)
    vec = vec && (out_dtype == LLMC_F32 || ((ldo % 8 == 0) && (((uintptr_t)out & 15) == 0)));
  else if (out_mode == LLMC_OUT_CODES)
    vec = vec && (ldo % 8 == 0) && (((uintptr_t)out & 7) == 0);
  else if (fmt == LLMC_FMT_FP4)
    vec = vec && (ldo % 4 == 0) && (((uintptr_t)out & 3) == 0);
  if (out_mode == LLMC_OUT_PACKED && fmt == LLMC_FMT_INT) {
    const int pf = 32 / p.bits;
    if (pf != 8 && pf != 4) {
      // fields are OR-ed into place: clear the destination first (a fill kernel, not a memset
      // node, so the call stays safe to capture in a HIP graph)
      const int64_t nw = R * ldo;
      hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, st, (uint32_t*)out, nw);
      LLMC_LAUNCH_STATUS();
    }
  }
  const int64_t threads = R * ((K + 7) / 8);
  const unsigned grid = (unsigned)((threads + 255) / 256);
  if (vec)
    hipLaunchKernelGGL((quantize_kernel<true>), dim3(grid), dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL((quantize_kernel<false>), dim3(grid), dim3(256), 0, st, p);
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int llmc_dynamic_per_token_quantize(const void* x, int32_t x_dtype, int64_t N, int64_t K,
                                               int64_t ldx, int32_t fmt, int32_t num_bits, int32_t out_mode,
                                               void* out, int64_t ldo, void* scale_out, void* stream) {
  LLMC_CHECK_ARG(x && N > 0 && K > 0, 1);
  LLMC_CHECK_ARG(x_dtype == LLMC_BF16 || x_dtype == LLMC_F16, 2);
  LLMC_CHECK_ARG(K <= 65536, 4);
  LLMC_CHECK_ARG(ldx >= K, 5);
  LLMC_CHECK_ARG(fmt == LLMC_FMT_INT || fmt == LLMC_FMT_FP8, 6);
  LLMC_CHECK_ARG(fmt != LLMC_FMT_INT || num_bits == 8, 7);
  LLMC_CHECK_ARG(out_mode == LLMC_OUT_FAKEQUANT || out_mode == LLMC_OUT_CODES, 8);
  LLMC_CHECK_ARG(out, 9);
  hipStream_t st = (hipStream_t)stream;
  const bool wave_ok = K % 8 == 0 && ldx % 8 == 0 && (((uintptr_t)x) & 15) == 0 &&
                       (out_mode == LLMC_OUT_CODES ? (ldo % 8 == 0 && (((uintptr_t)out) & 7) == 0)
                                                   : (ldo % 8 == 0 && (((uintptr_t)out) & 15) == 0));
  if (wave_ok) {
    const int nb = fmt == LLMC_FMT_INT ? num_bits : 8;
    if (x_dtype == LLMC_BF16)
      launch_token_wave_nc<LLMC_BF16>(x, ldx, N, (int)K, fmt, nb, out_mode, out, ldo, scale_out, st);
    else
      launch_token_wave_nc<LLMC_F16>(x, ldx, N, (int)K, fmt, nb, out_mode, out, ldo, scale_out, st);
    LLMC_LAUNCH_STATUS();
    return 0;
  }
  const size_t smem = (size_t)((K + 7) / 8 * 8) * 2;
  auto kern = x_dtype == LLMC_BF16 ? dynamic_token_kernel<LLMC_BF16> : dynamic_token_kernel<LLMC_F16>;
  if (smem > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (e != hipSuccess) return 1000 + (int)e;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)N), dim3(256), smem, st, x, ldx, (int)K, fmt,
                     fmt == LLMC_FMT_INT ? num_bits : 8, out_mode, out, ldo, scale_out);
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int llmc_dynamic_group_quantize(const void* x, int32_t x_dtype, int64_t N, int64_t K, int64_t ldx,
                                           int64_t group, int32_t fmt, int32_t num_bits, int32_t scale_mode,
                                           const float* global_scale, void* out, int64_t ldo, void* stream) {
  LLMC_CHECK_ARG(x && N > 0 && K > 0 && (((uintptr_t)x) & 15) == 0, 1);
  LLMC_CHECK_ARG(x_dtype == LLMC_BF16 || (x_dtype == LLMC_F16 && scale_mode != LLMC_SCALE_MXFP4), 2);
  LLMC_CHECK_ARG(K <= (1LL << 30) && units_fit(N, (K + 15) / 16), 4);
  LLMC_CHECK_ARG(ldx >= K && ldx % 8 == 0, 5);
  const int lg = log2_exact(group);
  LLMC_CHECK_ARG(lg >= 4 && lg <= 10 && K % group == 0, 6);
  LLMC_CHECK_ARG(fmt >= 0 && fmt <= 2, 7);
  LLMC_CHECK_ARG(fmt != LLMC_FMT_INT || num_bits == 4 || num_bits == 8, 8);
  LLMC_CHECK_ARG(scale_mode >= 0 && scale_mode <= 2 && (scale_mode == LLMC_SCALE_PLAIN || fmt == LLMC_FMT_FP4), 9);
  LLMC_CHECK_ARG(scale_mode != LLMC_SCALE_NVFP4 || global_scale, 10);
  LLMC_CHECK_ARG(out && (((uintptr_t)out) & 15) == 0 && ldo >= K && ldo % 8 == 0, 11);
  QuantParams p = {};
  p.x = x; p.x_dt = x_dtype; p.R = N; p.K = K; p.ldx = ldx;
  p.gscale = global_scale; p.fmt = fmt; p.bits = fmt == LLMC_FMT_INT ? num_bits : (fmt == LLMC_FMT_FP8 ? 8 : 4);
  p.out_mode = LLMC_OUT_FAKEQUANT; p.out = out; p.out_dt = x_dtype; p.ldo = ldo;
  RowsWalk w;
  walk_rows(w, N, K, 16);
  w.cshift = 31;
  w.rshift = 63;
  w.lanes = (int)(group / 16);
  const int sm = scale_mode == LLMC_SCALE_MXFP4 ? SM_OWN_MX : scale_mode == LLMC_SCALE_NVFP4 ? SM_OWN_NVFP4 : SM_OWN;
  if (x_dtype == LLMC_BF16)
    launch_rows_sm<LLMC_BF16>(sm, p, w, 16, (hipStream_t)stream);
  else
    launch_rows_sm<LLMC_F16>(sm, p, w, 16, (hipStream_t)stream);
  LLMC_LAUNCH_STATUS();
  return 0;
}
