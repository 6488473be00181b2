// MSE observer: grid search over shrink factors p_i = 1 - i/grid of each group's (min,max).
//
// The reference walks the steps on the host and stops GLOBALLY after `patience`
// consecutive steps in which no group improved.  Here every group walks all steps in
// one launch with its running best in registers and records the steps at which it
// improved in a bit mask; the masks are OR-ed into a global per-step flag word.  A
// last kernel replays the patience rule on the flags to get the stop step and picks,
// per group, its latest improvement at or before that step -- the same selection as
// the host loop, without a host round trip per step.  The inner loop is bound by
// vector instructions; the weight is read from HBM once.
#include <string.h>

#include <mutex>

#include "qformat.h"

namespace {

constexpr int MAX_STEPS = 256;
constexpr int MASK_WORDS = MAX_STEPS / 64;

struct MseParams {
  const void* x;
  int dt;            // dtype of the observed values (and of every intermediate)
  int fmt, bits, symmetric, scale_mode;
  int steps;
  double grid;       // step i shrinks the range by p_i = (float)(1.0 - i/grid), as the host loop does
  float norm;
  float expand;
  void* min0;        // [N] expanded observed min (dtype dt)
  void* max0;        // [N]
  uint64_t* masks;   // [N][mask_words(steps)]
  uint64_t* flags;   // [MASK_WORDS] zero-initialised
  const uint16_t* powtab;  // a^norm rounded to dt for every non-negative 16-bit a (see mse_setup_kernel), or NULL
  const float* factors;    // [steps] the steps' shrink factors
  // importance-weighted variant (observers/imatrix.py:255-328): the error |fq(x) - x|^norm is formed and
  // summed in fp32 (values are quantised in dt as before) and weighted per input channel
  int err32;
  const float* imp;  // [K] weights, or NULL for uniform
};

// words of a group's mask: one covers the usual searches (20 or 80 steps take one or four)
__host__ __device__ __forceinline__ int mask_words(int steps) { return steps <= 64 ? 1 : MASK_WORDS; }

__device__ __forceinline__ float step_factor(int i, double grid) { return (float)(1.0 - (double)i / grid); }

// a^norm (a >= 0) as the eager pow forms it in dtype dt: exponents 2, 3 and 0.5 have closed forms (a*a,
// (a*a)*a with the inner product rounded to dt as well, sqrt), anything else is one pow rounded to dt
__device__ __forceinline__ float pow_eager(float a, float norm, int dt) {
  if (norm == 2.0f) return round_rt(__fmul_rn(a, a), dt);
  if (norm == 3.0f) return round_rt(__fmul_rn(round_rt(__fmul_rn(a, a), dt), a), dt);
  if (norm == 0.5f) return round_rt(__fsqrt_rn(a), dt);
  return round_rt(powf(a, norm), dt);
}

// |fq(x) - x|^norm with every intermediate rounded to dt
__device__ __forceinline__ float elem_error(float x, float s, float zp, bool has_zp, int dt, const QFormat& f,
                                            float norm) {
  const float q = quantize_value(x, s, zp, has_zp, dt, f);
  const float dq = dequantize_value(q, s, zp, has_zp, dt);
  const float a = fabsf(round_rt(dq - x, dt));
  // `norm` arrives already rounded to dt: the eager pow converts its scalar exponent to the tensor dtype
  return pow_eager(a, norm, dt);
}

// fp32 error of the importance-weighted search: fq(x) in dt, then (fq - x), abs, pow in fp32; the
// eager pow multiplies for exponents 2 and 3
__device__ __forceinline__ float elem_error32(float x, float s, float zp, bool has_zp, int dt, const QFormat& f,
                                              float norm) {
  const float q = quantize_value(x, s, zp, has_zp, dt, f);
  const float dq = dequantize_value(q, s, zp, has_zp, dt);
  const float a = fabsf(__fsub_rn(dq, x));
  if (norm == 2.0f) return __fmul_rn(a, a);
  if (norm == 3.0f) return __fmul_rn(__fmul_rn(a, a), a);
  if (norm == 0.5f) return __fsqrt_rn(a);
  return powf(a, norm);
}

__device__ __forceinline__ void unpack8(uint4 v, int dt, float* o) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (dt == LLMC_BF16) {
      o[2 * j] = __uint_as_float(w[j] << 16);
      o[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    } else {
      o[2 * j] = f16_bits_to_f32((uint16_t)(w[j] & 0xffffu));
      o[2 * j + 1] = f16_bits_to_f32((uint16_t)(w[j] >> 16));
    }
  }
}

__device__ __forceinline__ void or_flags(uint64_t* flags, const uint64_t* m) {
  // OR over the workgroup first, then one atomic per word and workgroup
  __shared__ unsigned long long sflags[MASK_WORDS];
  if (threadIdx.x < MASK_WORDS) sflags[threadIdx.x] = 0ull;
  __syncthreads();
#pragma unroll
  for (int wd = 0; wd < MASK_WORDS; ++wd) {
    unsigned long long v = m[wd];
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicOr(&sflags[wd], v);
  }
  __syncthreads();
  if (threadIdx.x < MASK_WORDS && sflags[threadIdx.x]) atomicOr((unsigned long long*)&flags[threadIdx.x], sflags[threadIdx.x]);
}

// 16-bit inputs, groups of g = 8*L consecutive elements (L a power of two <= 64 lanes per group)
__global__ __launch_bounds__(256) void mse_team_kernel(MseParams p, int64_t ngroups, int ng, int g, int L,
                                                       int64_t ldw) {
  const int64_t gtid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t grp = gtid / L;
  const int sub = (int)(gtid % L);
  const bool live = grp < ngroups;
  const QFormat f = make_qformat(p.fmt, p.bits);
  float xv[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) xv[j] = 0.f;
  float mn = INFINITY, mx = -INFINITY;
  if (live) {
    const int64_t r = grp / ng, gi = grp % ng;
    const uint4 v = *(const uint4*)((const uint16_t*)p.x + r * ldw + gi * g + (int64_t)sub * 8);
    unpack8(v, p.dt, xv);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      mn = fminf(mn, xv[j]);
      mx = fmaxf(mx, xv[j]);
    }
  }
  for (int o = L >> 1; o > 0; o >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, o, 64));
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  }
  mn = round_rt(product<LLMC_F16>(mn, p.expand), p.dt);
  mx = round_rt(product<LLMC_F16>(mx, p.expand), p.dt);
  float best = p.dt == LLMC_BF16 ? 3.3895313892515355e38f : p.dt == LLMC_F16 ? 65504.0f : 3.4028234663852886e38f;
  if (p.err32) best = 3.4028234663852886e38f;
  float wt[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) wt[j] = 1.f;
  if (p.err32 && p.imp && live) {
    const int64_t gi = grp % ng;
#pragma unroll
    for (int j = 0; j < 8; ++j) wt[j] = p.imp[gi * g + (int64_t)sub * 8 + j];
  }
  uint64_t mask[MASK_WORDS];
#pragma unroll
  for (int wd = 0; wd < MASK_WORDS; ++wd) mask[wd] = 0ull;
  for (int i = 0; i < p.steps; ++i) {
    const float pi = step_factor(i, p.grid);
    const float smin = round_rt(product<LLMC_F16>(mn, pi), p.dt), smax = round_rt(product<LLMC_F16>(mx, pi), p.dt);
    float s, zp;
    int e;
    qparams_from_minmax(smin, smax, p.dt, f, p.symmetric != 0, p.scale_mode, 1.f, &s, &zp, &e);
    float err = 0.f;
    if (p.err32) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float ej = elem_error32(xv[j], s, zp, !p.symmetric, p.dt, f, p.norm);
        err += p.imp ? __fmul_rn(ej, wt[j]) : ej;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) err += elem_error(xv[j], s, zp, !p.symmetric, p.dt, f, p.norm);
    }
    for (int o = L >> 1; o > 0; o >>= 1) err += __shfl_xor(err, o, 64);
    if (!p.err32) err = round_rt(err, p.dt);
    if (err < best) {
      best = err;
#pragma unroll
      for (int wd = 0; wd < MASK_WORDS; ++wd)
        if (wd == (i >> 6)) mask[wd] |= 1ull << (i & 63);
    }
  }
  if (!live) {
#pragma unroll
    for (int wd = 0; wd < MASK_WORDS; ++wd) mask[wd] = 0ull;
  }
  if (live && sub == 0) {
    store_rt(p.min0, grp, mn, p.dt);
    store_rt(p.max0, grp, mx, p.dt);
#pragma unroll
    for (int wd = 0; wd < MASK_WORDS; ++wd)
      if (wd < mask_words(p.steps)) p.masks[grp * mask_words(p.steps) + wd] = mask[wd];
  }
  or_flags(p.flags, mask);
}

// ---- 16-bit inputs: the same arithmetic with everything the format decides fixed at compile time.  Per element and
// candidate the search has to round the quotient, quantise, scale back, round, subtract, round, look the power up and
// add; what is done on top is kept off that path:
//   - x / s needs one multiply (bf16) or three operations (f16) to round correctly (quot16), with one range check per
//     lane and one per candidate instead of a guard per element;
//   - roundings go through the packed conversion, two elements at a time;
//   - a is a 16-bit value, so a^norm rounded to the dtype is a lookup in a 32768-entry table (64 KiB of LDS);
//   - shrink factors are computed once per call (a double division per lane and candidate before);
//   - a candidate whose scale rounds to the previous one's has the previous one's error and cannot improve on it, so
//     it is skipped: MXFP4's power-of-two scales leave one or two distinct candidates of twenty;
//   - two 8-element chunks per lane share the candidate's scale arithmetic.
// Sums keep the order they always had (8 elements, then the lanes by descending distance), so near-ties between
// candidates fall as before.  NVFP4 groups of a 14336 x 4096 weight, 20 candidates, with the launches around it: 1036 -> 533 us; MXFP4 1057 -> 162 us.

template <int DT>
__device__ __forceinline__ void unpack2(uint32_t w, float& lo, float& hi) {
  if (DT == LLMC_BF16) {
    lo = __uint_as_float(w << 16);
    hi = __uint_as_float(w & 0xffff0000u);
  } else {
    lo = f16_bits_to_f32((uint16_t)(w & 0xffffu));
    hi = f16_bits_to_f32((uint16_t)(w >> 16));
  }
}
template <int DT>
__device__ __forceinline__ void unpack8t(const uint4& v, float* x) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) unpack2<DT>(w[j], x[2 * j], x[2 * j + 1]);
}

// both values rounded to DT
template <int DT>
__device__ __forceinline__ void round_pair(float& a, float& b) {
  unpack2<DT>(pack16<DT>(a, b), a, b);
}

// a^norm (a >= 0) rounded to DT.  a = m*2^E; norm*E is exact in fp32 (norm has at most 11
// significant bits, E at most 8) and splits into an integer I and a fraction r, so
// a^norm = 2^I * 2^(r + norm*log2 m) with the second exponent small: the hardware log2/exp2 (1 ulp
// each) leave a few ulps of error in total.  If rounding to DT could fall either way within 16 ulps
// the library powf decides, so the rounded value matches the reference's pow-then-round.
template <int DT>
__device__ __forceinline__ float pow_round16(float a, float norm) {
  const float m = __builtin_amdgcn_frexp_mantf(a);
  const int E = __builtin_amdgcn_frexp_expf(a);
  const float y = norm * (float)E;
  const float I = rintf(y);
  const float t = fmaf(norm, __builtin_amdgcn_logf(m), y - I);
  const float pf = ldexpf(__builtin_amdgcn_exp2f(t), (int)I);
  const uint32_t w = pack16<DT>(pf * 0.99999809265136719f, pf * 1.0000019073486328f);  // 1 -+ 2^-19
  if ((w & 0xffffu) != (w >> 16)) return round_rt(powf(a, norm), DT);
  return DT == LLMC_BF16 ? __uint_as_float(w << 16) : f16_bits_to_f32((uint16_t)(w & 0xffffu));
}

// values or a scale outside the ranges of quot16: the plain division
template <int DT, int FMT, bool HAS_ZP>
__device__ __attribute__((noinline)) float elem_error_plain(float x, float s, float zp, int bits, float norm) {
  return elem_error(x, s, zp, HAS_ZP, DT, make_qformat(FMT, bits), norm);
}

// err + |fq(x) - x|^norm over N elements in order, every intermediate rounded to DT.  `plain`: quot16 applies.
template <int DT, int FMT, bool HAS_ZP, bool TAB, int N>
__device__ __forceinline__ float chunk_error(float err, const float (&x)[N], const FastDiv& d, float zp,
                                             const QFormat& f, int bits, float norm, bool plain,
                                             const uint16_t* __restrict__ tab) {
  const float s = d.s;
  if (!plain) {
#pragma unroll 1
    for (int j = 0; j < N; ++j) err += elem_error_plain<DT, FMT, HAS_ZP>(x[j], s, zp, bits, norm);
    return err;
  }
  uint32_t aw[N / 2];  // the errors a as packed 16-bit values, signs undefined
#pragma unroll
  for (int j = 0; j < N / 2; ++j) {
    float v0 = quot16<DT>(x[2 * j], d), v1 = quot16<DT>(x[2 * j + 1], d);
    if (FMT == LLMC_FMT_FP4) {
      // rounded to DT, then to e2m1 straight from the packed pair (the conversion saturates at 6 by itself)
      const f32x2_t t = hw_e2m1_pair_decode(hw_e2m1_pair16<DT>(pack16<DT>(v0, v1)));
      v0 = t.x * s;
      v1 = t.y * s;
      round_pair<DT>(v0, v1);
      aw[j] = pack16<DT>(v0 - x[2 * j], v1 - x[2 * j + 1]);
      continue;
    }
    round_pair<DT>(v0, v1);
    if (HAS_ZP) {
      v0 += zp;
      v1 += zp;
      round_pair<DT>(v0, v1);
    }
    // (the sign of a zero quotient does not reach |fq(x) - x|, so the reference's added zero is left out)
    v0 = __builtin_amdgcn_fmed3f(v0, f.qmin, f.qmax);
    v1 = __builtin_amdgcn_fmed3f(v1, f.qmin, f.qmax);
    if (FMT == LLMC_FMT_INT) {
      v0 = rintf(v0);
      v1 = rintf(v1);
    } else {
      const f32x2_t t = hw_e4m3_pair_decode(hw_e4m3_pair(v0, v1));
      v0 = t.x;
      v1 = t.y;
    }
    if (HAS_ZP) {
      v0 -= zp;
      v1 -= zp;
      round_pair<DT>(v0, v1);
    }
    v0 *= s;
    v1 *= s;
    round_pair<DT>(v0, v1);
    aw[j] = pack16<DT>(v0 - x[2 * j], v1 - x[2 * j + 1]);
  }
  if (TAB) {
    uint32_t pw[N];
#pragma unroll
    for (int j = 0; j < N / 2; ++j) {  // byte offsets of the two table entries
      pw[2 * j] = *(const uint16_t*)((const char*)tab + ((aw[j] << 1) & 0xfffeu));
      pw[2 * j + 1] = *(const uint16_t*)((const char*)tab + ((aw[j] >> 15) & 0xfffeu));
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
      err += DT == LLMC_BF16 ? __uint_as_float(pw[j] << 16) : f16_bits_to_f32((uint16_t)pw[j]);
    return err;
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const uint16_t bits16 = (uint16_t)((j & 1 ? aw[j >> 1] >> 16 : aw[j >> 1]) & 0x7fffu);
    const float a = DT == LLMC_BF16 ? bf16_bits_to_f32(bits16) : f16_bits_to_f32(bits16);
    if (norm == 2.0f)
      err += round16_finite<DT>(a * a);
    else if (norm == 3.0f)
      err += round16_finite<DT>(round16_finite<DT>(a * a) * a);
    else if (norm == 0.5f)
      err += round16_finite<DT>(__fsqrt_rn(a));
    else
      err += pow_round16<DT>(a, norm);
  }
  return err;
}

// v + the value of the lane at distance O (a power of two below 16)
template <int O>
__device__ __forceinline__ float add_xor(float v) {
  if constexpr (O == 1 || O == 2) {  // inside a quad: a data-parallel move
    constexpr int perm = O == 1 ? 0xB1 : 0x4E;
    return v + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), perm, 0xf, 0xf, true));
  } else {
    return v + __shfl_xor(v, O, 64);
  }
}

// How a group's candidate scales follow from its (expanded) range.  Symmetric: from the largest magnitude alone, one
// product and one division by the format's constant half range per candidate.
enum { RULE_ASYM = 0, RULE_SYM = 1, RULE_SYM_MX = 2 };
template <int DT, int FMT, int RULE>
struct StepScale {
  float mn, mx, amax, half, rhalf;
  bool corrected;  // the quotient by three operations is the IEEE one
  const QFormat f;
  __device__ __forceinline__ StepScale(float lo, float hi, const QFormat& fmt) : mn(lo), mx(hi), f(fmt) {
    amax = fmaxf(-fminf(lo, 0.f), fmaxf(hi, 0.f));
    half = (f.qmax - f.qmin) * 0.5f;
    rhalf = __fdiv_rn(1.0f, half);
    corrected = amax > 0x1p-60f && amax < 0x1p60f;
  }
  __device__ __forceinline__ void at(float factor, float* s, float* zp) const {
    if (RULE == RULE_SYM) {
      const float a = round16_finite<DT>(product<DT>(amax, factor));
      float q;
      if (corrected) {  // rhalf is correctly rounded, so one residual step gives the correctly rounded quotient
        q = a * rhalf;
        q = fmaf(fmaf(-half, q, a), rhalf, q);
      } else {
        q = a / half;
      }
      q = round16_finite<DT>(q);
      *s = q == 0.f ? dtype_eps(DT) : q;
      *zp = 0.f;
      return;
    }
    if (RULE == RULE_SYM_MX && DT == LLMC_BF16) {
      // the exponent field of the bf16 magnitude, raised by half an e2m1 step, less emax = 2 (qparams_from_minmax)
      const uint32_t a = (__float_as_uint(round16_finite<DT>(amax * factor)) >> 16) + 32u;
      const uint32_t e = (a >> 7) & 0xffu;
      if (e > 2u && e < 255u) {
        *s = __uint_as_float((e - 2u) << 23);
        *zp = 0.f;
        return;
      }
    }
    int e;
    qparams_from_minmax(round_to<DT>(product<DT>(mn, factor)), round_to<DT>(product<DT>(mx, factor)), DT, f, RULE != RULE_ASYM,
                        RULE == RULE_SYM_MX ? LLMC_SCALE_MXFP4 : LLMC_SCALE_PLAIN, 1.f, s, zp, &e);
  }
};

template <int DT>
__device__ __forceinline__ float largest_finite() {
  return DT == LLMC_BF16 ? 3.3895313892515355e38f : 65504.0f;
}

// the table into LDS (64 KiB), by the whole workgroup; no other use of LDS before the barrier
__device__ __forceinline__ void load_powtab(uint16_t* lds, const uint16_t* tab) {
  const uint4* src = (const uint4*)tab;
  uint4* dst = (uint4*)lds;
#pragma unroll 4
  for (int k = threadIdx.x; k < 65536 / 16; k += blockDim.x) dst[k] = src[k];
}

// Groups of g = 8 * C * L consecutive elements: L (a power of two <= 32) neighbouring lanes with C chunks of 8 each
// (C = 2, or 1 for groups of 8).  TAB: the power comes from p.powtab through LDS, in workgroups of 1024 threads of which
// two fill a CU (its LDS and its waves); a workgroup walks over the groups in strides of the grid (what the chip holds at once), so that
// the table is fetched 512 times per call at most.
constexpr int TEAM_BLOCK = 1024;
template <int DT, int FMT, int RULE, bool TAB, int C, int MW>
__global__ __launch_bounds__(TAB ? TEAM_BLOCK : 256) void mse_team_fast_kernel(MseParams p, int64_t ngroups, int ng, int g,
                                                                        int lshift, int64_t ldw) {
  const int BLOCK = TAB ? blockDim.x : 256;
  extern __shared__ __attribute__((aligned(16))) uint16_t powlds[];
  if (TAB) load_powtab(powlds, p.powtab);
  constexpr bool SYM = RULE != RULE_ASYM;
  __shared__ float factors[MW * 64];
  if (threadIdx.x < MW * 64) factors[threadIdx.x] = (int)threadIdx.x < p.steps ? p.factors[threadIdx.x] : 0.f;  // <= 256
  __syncthreads();
  const int L = 1 << lshift;
  const QFormat f = make_qformat(FMT, p.bits);
  uint64_t any[MASK_WORDS];  // OR of this thread's masks over its groups
#pragma unroll
  for (int wd = 0; wd < MASK_WORDS; ++wd) any[wd] = 0ull;
  const int64_t threads = ngroups << lshift;
  // the bound is uniform over the workgroup and a group's lanes branch alike, so they meet in every exchange
  for (int64_t base = (int64_t)blockIdx.x * BLOCK; base < threads; base += (int64_t)gridDim.x * BLOCK) {
    const int64_t gtid = base + threadIdx.x;
    const int64_t grp = gtid >> lshift;
    const int sub = (int)(gtid & (L - 1));
    const bool live = grp < ngroups;
    float xv[C][8];
    float mn = INFINITY, mx = -INFINITY;
    ValueRange<DT> range;
#pragma unroll
    for (int k = 0; k < C; ++k) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (live) {
        const int64_t r = grp / ng, gi = grp % ng;
        v = *(const uint4*)((const uint16_t*)p.x + r * ldw + gi * g + (int64_t)(sub * C + k) * 8);
      }
      range.add(v);
      unpack8t<DT>(v, xv[k]);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        mn = fminf(mn, xv[k][j]);
        mx = fmaxf(mx, xv[k][j]);
      }
    }
    for (int o = L >> 1; o > 0; o >>= 1) {
      mn = fminf(mn, __shfl_xor(mn, o, 64));
      mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    }
    mn = round_to<DT>(product<DT>(mn, p.expand));
    mx = round_to<DT>(product<DT>(mx, p.expand));
    const bool values_plain = range.plain();
    float best = largest_finite<DT>();
    uint64_t mask[MW];
#pragma unroll
    for (int wd = 0; wd < MW; ++wd) mask[wd] = 0ull;
    const StepScale<DT, FMT, RULE> scales(mn, mx, f);
    float s_prev = -1.f;
    for (int i = 0; live; ++i) {
      float s = 0.f, zp = 0.f;
      for (; i < p.steps; ++i) {  // the next candidate with a scale of its own
        scales.at(factors[i], &s, &zp);
        if (!SYM || s != s_prev) break;
      }
      if (i >= p.steps) break;
      s_prev = s;
      const FastDiv d = make_fastdiv(s);
      const bool plain = values_plain && scale_plain<DT>(s);
      float err[C];
#pragma unroll
      for (int k = 0; k < C; ++k)
        err[k] = chunk_error<DT, FMT, !SYM, TAB, 8>(0.f, xv[k], d, zp, f, p.bits, p.norm, plain, powlds);
      // lanes of 8 elements by descending distance; the last step joins a lane's own two chunks
      switch (lshift) {
        case 5:
#pragma unroll
          for (int k = 0; k < C; ++k) err[k] += __shfl_xor(err[k], 16, 64);
          [[fallthrough]];
        case 4:
#pragma unroll
          for (int k = 0; k < C; ++k) err[k] = add_xor<8>(err[k]);
          [[fallthrough]];
        case 3:
#pragma unroll
          for (int k = 0; k < C; ++k) err[k] = add_xor<4>(err[k]);
          [[fallthrough]];
        case 2:
#pragma unroll
          for (int k = 0; k < C; ++k) err[k] = add_xor<2>(err[k]);
          [[fallthrough]];
        case 1:
#pragma unroll
          for (int k = 0; k < C; ++k) err[k] = add_xor<1>(err[k]);
          break;
        default: break;
      }
      const float e = round_to<DT>(C == 2 ? err[0] + err[C - 1] : err[0]);
      if (e < best) {
        best = e;
#pragma unroll
        for (int wd = 0; wd < MW; ++wd)
          if (MW == 1 || wd == (i >> 6)) mask[wd] |= 1ull << (i & 63);
      }
    }
    if (live && sub == 0) {
      store_from_f32<DT>(p.min0, grp, mn);
      store_from_f32<DT>(p.max0, grp, mx);
#pragma unroll
      for (int wd = 0; wd < MW; ++wd) p.masks[grp * MW + wd] = mask[wd];
    }
#pragma unroll
    for (int wd = 0; wd < MW; ++wd) any[wd] |= mask[wd];
  }
  or_flags(p.flags, any);
}

// Once per call: the flag words cleared, the steps' shrink factors, and (fill_tab) a^norm rounded to dt for each of the
// 32768 non-negative 16-bit values a, as 16-bit patterns -- exactly what the eager pow gives element by element.
__global__ __launch_bounds__(256) void mse_setup_kernel(uint64_t* flags, float* factors, int steps, double grid,
                                                        uint16_t* __restrict__ tab, int fill_tab, float norm, int dt) {
  if (blockIdx.x == 0) {
    if (threadIdx.x < MASK_WORDS) flags[threadIdx.x] = 0ull;
    if ((int)threadIdx.x < steps) factors[threadIdx.x] = step_factor(threadIdx.x, grid);
  }
  if (!fill_tab) return;
  const int i = blockIdx.x * 256 + threadIdx.x;
  const float a = dt == LLMC_BF16 ? bf16_bits_to_f32((uint16_t)i) : f16_bits_to_f32((uint16_t)i);
  const float r = pow_eager(a, norm, dt);
  tab[i] = dt == LLMC_BF16 ? f32_to_bf16_bits(r) : f32_to_f16_bits(r);
}

template <class Kernel>
int allow_lds(Kernel kern, int bytes) {
  const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  return e == hipSuccess ? 0 : 1000 + (int)e;
}

template <int DT, int FMT, int RULE, int C, int MW>
int launch_team_words(const MseParams& p, int64_t n, int ng, int g, int lshift, int64_t ldw, hipStream_t st) {
  const int64_t threads = n << lshift;
  if (p.powtab != nullptr) {
    auto kern = mse_team_fast_kernel<DT, FMT, RULE, true, C, MW>;
    static const int configured = allow_lds(kern, 65536);
    if (configured) return configured;
    // small calls: workgroups of 256 while those leave CUs without any
    const int block = threads <= 256 * 256 ? 256 : TEAM_BLOCK;
    const int64_t wgs = (threads + block - 1) / block;
    hipLaunchKernelGGL(kern, dim3((unsigned)(wgs < 512 ? wgs : 512)), dim3(block), 65536, st, p, n, ng, g, lshift, ldw);
  } else {
    const int64_t wgs = (threads + 255) / 256;
    hipLaunchKernelGGL((mse_team_fast_kernel<DT, FMT, RULE, false, C, MW>), dim3((unsigned)(wgs < 8192 ? wgs : 8192)),
                       dim3(256), 0, st, p, n, ng, g, lshift, ldw);
  }
  return 0;
}

// one word of candidates in the usual searches (20 or 80 steps), all four beyond
template <int DT, int FMT, int RULE, int C>
int launch_team_chunks(const MseParams& p, int64_t n, int ng, int g, int lshift, int64_t ldw, hipStream_t st) {
  return p.steps <= 64 ? launch_team_words<DT, FMT, RULE, C, 1>(p, n, ng, g, lshift, ldw, st)
                       : launch_team_words<DT, FMT, RULE, C, MASK_WORDS>(p, n, ng, g, lshift, ldw, st);
}

template <int DT, int FMT, int RULE>
int launch_team_fast_one(const MseParams& p, int64_t n, int ng, int g, int lshift, int64_t ldw, hipStream_t st) {
  return lshift == 0 ? launch_team_chunks<DT, FMT, RULE, 1>(p, n, ng, g, 0, ldw, st)
                     : launch_team_chunks<DT, FMT, RULE, 2>(p, n, ng, g, lshift - 1, ldw, st);
}

template <int DT>
int launch_team_fast(const MseParams& p, int64_t n, int ng, int g, int lshift, int64_t ldw, hipStream_t st) {
  if (p.fmt == LLMC_FMT_INT)
    return p.symmetric ? launch_team_fast_one<DT, LLMC_FMT_INT, RULE_SYM>(p, n, ng, g, lshift, ldw, st)
                       : launch_team_fast_one<DT, LLMC_FMT_INT, RULE_ASYM>(p, n, ng, g, lshift, ldw, st);
  if (p.fmt == LLMC_FMT_FP8)
    return p.symmetric ? launch_team_fast_one<DT, LLMC_FMT_FP8, RULE_SYM>(p, n, ng, g, lshift, ldw, st)
                       : launch_team_fast_one<DT, LLMC_FMT_FP8, RULE_ASYM>(p, n, ng, g, lshift, ldw, st);
  if (p.scale_mode == LLMC_SCALE_MXFP4)
    return launch_team_fast_one<DT, LLMC_FMT_FP4, RULE_SYM_MX>(p, n, ng, g, lshift, ldw, st);
  return launch_team_fast_one<DT, LLMC_FMT_FP4, RULE_SYM>(p, n, ng, g, lshift, ldw, st);
}

struct GenericLayout {
  int mode;  // 0: (n0, n1, G) view with element strides (s0, s1, 1); 1: bh x bw blocks of an [R,K] matrix
  int64_t n0, G, s0, s1;
  int R, K, bh, bw, nbc;
  int bshift;  // log2(bw), or -1
  int64_t ldw;
  int64_t ng;  // mode 0, weighted search: groups per row (column of element e of group n1 = (n1 % ng)*G + e % G)
};

__device__ __forceinline__ float generic_load(const void* x, int dt, const GenericLayout& l, int64_t n1, int64_t e) {
  if (l.mode == 0) return load_rt(x, (e / l.G) * l.s0 + n1 * l.s1 + (e % l.G), dt);
  const int br = (int)(n1 / l.nbc), bc = (int)(n1 % l.nbc);
  const int rr = br * l.bh + (int)(e / l.bw), cc = bc * l.bw + (int)(e % l.bw);
  return (rr < l.R && cc < l.K) ? load_rt(x, (int64_t)rr * l.ldw + cc, dt) : 0.f;
}

__device__ __forceinline__ float block_sum(float v, float* sh) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  return sh[0] + sh[1] + sh[2] + sh[3];
}

// Long groups of 16-bit values (a channel, a 128 x 128 block, a group that is no power of two): 256 threads per group,
// thread t holding the elements t, t + 256, ... in registers, packed in pairs, NV of them at most.  A candidate's error
// is summed per thread in element order, over the wavefront by descending distance and over the four wavefronts in
// order, as mse_generic_kernel does, but the wavefronts' sums wait in LDS until all candidates are through: no barrier
// per candidate.  The values were re-read and re-divided in full at every candidate before: FP8 channels of a
// 4061 x 14200 weight, 20 candidates, 6.1 ms -> 0.76 ms.
constexpr int ROW_THREADS = 256;
template <int DT, int FMT, int RULE, bool TAB, int NV, int UNITS>
__global__ __launch_bounds__(ROW_THREADS* UNITS, 4) void mse_rows_fast_kernel(MseParams p, GenericLayout l, int64_t n) {
  extern __shared__ __attribute__((aligned(16))) uint16_t powlds[];  // TAB: 64 KiB, then the partial sums
  float* sums = (float*)((char*)powlds + (TAB ? 65536 : 0));         // [UNITS][steps][4]
  __shared__ float shm[UNITS][8];
  if (TAB) load_powtab(powlds, p.powtab);
  constexpr bool SYM = RULE != RULE_ASYM;
  constexpr int N = NV < 8 ? NV : 8;  // elements per chunk of work
  const int unit = threadIdx.x / ROW_THREADS, t = threadIdx.x % ROW_THREADS, wave = t >> 6;
  float* mine = sums + unit * p.steps * 4;
  const QFormat f = make_qformat(FMT, p.bits);
  const int total = (int)(l.mode == 0 ? l.n0 * l.G : (int64_t)l.bh * l.bw);
  uint64_t any[MASK_WORDS];
#pragma unroll
  for (int wd = 0; wd < MASK_WORDS; ++wd) any[wd] = 0ull;
  for (int64_t base = (int64_t)blockIdx.x * UNITS; base < n; base += (int64_t)gridDim.x * UNITS) {
    const int64_t n1 = base + unit;
    const bool live = n1 < n;
    uint32_t xp[NV / 2];
    float mn = INFINITY, mx = -INFINITY;
    ValueRange<DT> range;
    // element e of the group: a contiguous run, or the rows of a block (0 past the matrix's edges)
    const int br = l.mode ? (int)(n1 / l.nbc) * l.bh : 0, bc = l.mode ? (int)(n1 % l.nbc) * l.bw : 0;
    const uint16_t* x = (const uint16_t*)p.x + (l.mode ? br * l.ldw + bc : n1 * l.s1);
    uint32_t first = t;
    asm volatile("" : "+v"(first));  // where each element lies is worked out here, not kept in registers over all groups
    auto load = [&](uint32_t e) -> uint32_t {
      if (!live || (int)e >= total) return 0u;
      if (l.mode == 0) return x[e];
      const uint32_t r = l.bshift >= 0 ? e >> l.bshift : e / (uint32_t)l.bw, c = e - r * (uint32_t)l.bw;
      return br + (int)r < l.R && bc + (int)c < l.K ? x[r * l.ldw + c] : 0u;
    };
#pragma unroll
    for (int k = 0; k < NV; k += 2) {
      xp[k / 2] = load(first + k * ROW_THREADS) | (load(first + (k + 1) * ROW_THREADS) << 16);
      if (k % 16 == 14) __builtin_amdgcn_sched_barrier(0);  // sixteen loads in flight, not the registers of them all
    }
#pragma unroll
    for (int k = 0; k < NV; k += 2) {
      float lo = 0.f, hi = 0.f;
      unpack2<DT>(xp[k / 2], lo, hi);
      range.add(xp[k / 2]);
      if (t + k * ROW_THREADS < total) {
        mn = fminf(mn, lo);
        mx = fmaxf(mx, lo);
      }
      if (t + (k + 1) * ROW_THREADS < total) {
        mn = fminf(mn, hi);
        mx = fmaxf(mx, hi);
      }
    }
    mn = wave_min(mn);
    mx = wave_max(mx);
    if ((t & 63) == 0) {
      shm[unit][wave] = mn;
      shm[unit][4 + wave] = mx;
    }
    __syncthreads();  // (also the table, the first time)
    mn = fminf(fminf(shm[unit][0], shm[unit][1]), fminf(shm[unit][2], shm[unit][3]));
    mx = fmaxf(fmaxf(shm[unit][4], shm[unit][5]), fmaxf(shm[unit][6], shm[unit][7]));
    mn = round_to<DT>(product<DT>(mn, p.expand));
    mx = round_to<DT>(product<DT>(mx, p.expand));
    const bool values_plain = range.plain();
    const StepScale<DT, FMT, RULE> scales(mn, mx, f);
    float s_prev = -1.f;
    for (int i = 0; i < p.steps; ++i) {
      float s, zp;
      scales.at(p.factors[i], &s, &zp);
      if (SYM && s == s_prev) {  // the previous candidate's error again
        if ((t & 63) == 0) mine[i * 4 + wave] = mine[(i - 1) * 4 + wave];
        continue;
      }
      s_prev = s;
      const FastDiv d = make_fastdiv(s);
      const bool plain = values_plain && scale_plain<DT>(s);
      float err = 0.f;
      // (elements past the end are zeros, whose error is an exact zero)
#pragma unroll
      for (int k = 0; k < NV; k += N) {
        // the values stay packed from one candidate to the next: unpacked once, 64 of them would fill the registers
        float xv[N];
#pragma unroll
        for (int j = 0; j < N; j += 2) {
          uint32_t w = xp[(k + j) / 2];
          asm volatile("" : "+v"(w));
          unpack2<DT>(w, xv[j], xv[j + 1]);
        }
        if (k % 16 == 0) __builtin_amdgcn_sched_barrier(0);
        if (plain || t + k * ROW_THREADS < total)
          err = chunk_error<DT, FMT, !SYM, TAB, N>(err, xv, d, zp, f, p.bits, p.norm, plain, powlds);
      }
      err += __shfl_xor(err, 32, 64);
      err += __shfl_xor(err, 16, 64);
      err = add_xor<8>(err);
      err = add_xor<4>(err);
      err = add_xor<2>(err);
      err = add_xor<1>(err);
      if ((t & 63) == 0) mine[i * 4 + wave] = err;
    }
    __syncthreads();
    if (t == 0 && live) {
      float best = largest_finite<DT>();
      uint64_t mask[MASK_WORDS];
#pragma unroll
      for (int wd = 0; wd < MASK_WORDS; ++wd) mask[wd] = 0ull;
      for (int i = 0; i < p.steps; ++i) {
        const float e = round_to<DT>(mine[i * 4] + mine[i * 4 + 1] + mine[i * 4 + 2] + mine[i * 4 + 3]);
        if (e < best) {
          best = e;
#pragma unroll
          for (int wd = 0; wd < MASK_WORDS; ++wd)
            if (wd == (i >> 6)) mask[wd] |= 1ull << (i & 63);
        }
      }
      store_from_f32<DT>(p.min0, n1, mn);
      store_from_f32<DT>(p.max0, n1, mx);
#pragma unroll
      for (int wd = 0; wd < MASK_WORDS; ++wd) {
        if (wd < mask_words(p.steps)) p.masks[n1 * mask_words(p.steps) + wd] = mask[wd];
        any[wd] |= mask[wd];
      }
    }
    __syncthreads();  // `mine` and `shm` are free again
  }
  or_flags(p.flags, any);
}

// Two groups per workgroup share one copy of the table where there are groups enough to fill the chip that way.
template <int DT, int FMT, int RULE, bool TAB, int NV, int UNITS>
int launch_rows(const MseParams& p, const GenericLayout& l, int64_t n, hipStream_t st) {
  constexpr int table = TAB ? 65536 : 0;
  auto kern = mse_rows_fast_kernel<DT, FMT, RULE, TAB, NV, UNITS>;
  static const int configured = allow_lds(kern, table + UNITS * MAX_STEPS * 16);
  if (configured) return configured;
  const int64_t wgs = (n + UNITS - 1) / UNITS;
  const dim3 grid((unsigned)(TAB && wgs > 512 ? 512 : wgs > 65536 ? 65536 : wgs));
  hipLaunchKernelGGL(kern, grid, dim3(UNITS * ROW_THREADS), table + UNITS * p.steps * 16, st, p, l, n);
  return 0;
}

template <int DT, int FMT, int RULE, bool TAB, int NV>
int launch_rows_units(const MseParams& p, const GenericLayout& l, int64_t n, hipStream_t st) {
  if constexpr (TAB)
    if (n >= 1024) return launch_rows<DT, FMT, RULE, TAB, NV, 2>(p, l, n, st);
  return launch_rows<DT, FMT, RULE, TAB, NV, 1>(p, l, n, st);
}

template <int DT, int FMT, int RULE>
int launch_rows_fast_one(const MseParams& p, const GenericLayout& l, int64_t n, int total, hipStream_t st) {
  const int nv = (total + ROW_THREADS - 1) / ROW_THREADS;
  if (!p.powtab)  // exponents with a closed form (2, 3, 0.5)
    return nv <= 8 ? launch_rows_units<DT, FMT, RULE, false, 8>(p, l, n, st)
                   : launch_rows_units<DT, FMT, RULE, false, 64>(p, l, n, st);
  if (nv <= 2) return launch_rows_units<DT, FMT, RULE, true, 2>(p, l, n, st);
  if (nv <= 4) return launch_rows_units<DT, FMT, RULE, true, 4>(p, l, n, st);
  if (nv <= 8) return launch_rows_units<DT, FMT, RULE, true, 8>(p, l, n, st);
  if (nv <= 24) return launch_rows_units<DT, FMT, RULE, true, 24>(p, l, n, st);
  return launch_rows_units<DT, FMT, RULE, true, 64>(p, l, n, st);
}

constexpr int ROWS_FAST_MAX = 64 * ROW_THREADS;

// does mse_rows_fast_kernel take this call?  (the weighted fp32 search, fp32 values and longer groups do not)
bool rows_fast_ok(const MseParams& p, int64_t total) {
  return p.dt != LLMC_F32 && !p.err32 && total <= ROWS_FAST_MAX && p.steps > 0 && (p.fmt != LLMC_FMT_FP4 || p.symmetric);
}

template <int DT>
int launch_rows_fast(const MseParams& p, const GenericLayout& l, int64_t n, int total, hipStream_t st) {
  if (p.fmt == LLMC_FMT_INT)
    return p.symmetric ? launch_rows_fast_one<DT, LLMC_FMT_INT, RULE_SYM>(p, l, n, total, st)
                       : launch_rows_fast_one<DT, LLMC_FMT_INT, RULE_ASYM>(p, l, n, total, st);
  if (p.fmt == LLMC_FMT_FP8)
    return p.symmetric ? launch_rows_fast_one<DT, LLMC_FMT_FP8, RULE_SYM>(p, l, n, total, st)
                       : launch_rows_fast_one<DT, LLMC_FMT_FP8, RULE_ASYM>(p, l, n, total, st);
  if (p.scale_mode == LLMC_SCALE_MXFP4)
    return launch_rows_fast_one<DT, LLMC_FMT_FP4, RULE_SYM_MX>(p, l, n, total, st);
  return launch_rows_fast_one<DT, LLMC_FMT_FP4, RULE_SYM>(p, l, n, total, st);
}

// any layout / dtype: one workgroup per group, values re-read (from L2) at every step
__global__ __launch_bounds__(256) void mse_generic_kernel(MseParams p, GenericLayout l) {
  __shared__ float sh[4];
  __shared__ float shm[8];
  const int64_t n1 = blockIdx.x;
  const int64_t total = l.mode == 0 ? l.n0 * l.G : (int64_t)l.bh * l.bw;
  const QFormat f = make_qformat(p.fmt, p.bits);
  float mn = INFINITY, mx = -INFINITY;
  for (int64_t e = threadIdx.x; e < total; e += 256) {
    const float v = generic_load(p.x, p.dt, l, n1, e);
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) {
    shm[threadIdx.x >> 6] = mn;
    shm[4 + (threadIdx.x >> 6)] = mx;
  }
  __syncthreads();
  mn = fminf(fminf(shm[0], shm[1]), fminf(shm[2], shm[3]));
  mx = fmaxf(fmaxf(shm[4], shm[5]), fmaxf(shm[6], shm[7]));
  mn = round_rt(product<LLMC_F16>(mn, p.expand), p.dt);
  mx = round_rt(product<LLMC_F16>(mx, p.expand), p.dt);
  float best = p.dt == LLMC_BF16 ? 3.3895313892515355e38f : p.dt == LLMC_F16 ? 65504.0f : 3.4028234663852886e38f;
  if (p.err32) best = 3.4028234663852886e38f;
  uint64_t mask[MASK_WORDS];
#pragma unroll
  for (int wd = 0; wd < MASK_WORDS; ++wd) mask[wd] = 0ull;
  for (int i = 0; i < p.steps; ++i) {
    const float pi = step_factor(i, p.grid);
    const float smin = round_rt(product<LLMC_F16>(mn, pi), p.dt), smax = round_rt(product<LLMC_F16>(mx, pi), p.dt);
    float s, zp;
    int e_;
    qparams_from_minmax(smin, smax, p.dt, f, p.symmetric != 0, p.scale_mode, 1.f, &s, &zp, &e_);
    float err = 0.f;
    if (p.err32) {
      for (int64_t e = threadIdx.x; e < total; e += 256) {
        const float ej = elem_error32(generic_load(p.x, p.dt, l, n1, e), s, zp, !p.symmetric, p.dt, f, p.norm);
        err += p.imp ? __fmul_rn(ej, p.imp[(n1 % l.ng) * l.G + e % l.G]) : ej;
      }
      err = block_sum(err, sh);
    } else {
      for (int64_t e = threadIdx.x; e < total; e += 256)
        err += elem_error(generic_load(p.x, p.dt, l, n1, e), s, zp, !p.symmetric, p.dt, f, p.norm);
      err = round_rt(block_sum(err, sh), p.dt);
    }
    if (err < best) {
      best = err;
#pragma unroll
      for (int wd = 0; wd < MASK_WORDS; ++wd)
        if (wd == (i >> 6)) mask[wd] |= 1ull << (i & 63);
    }
  }
  if (threadIdx.x == 0) {
    store_rt(p.min0, n1, mn, p.dt);
    store_rt(p.max0, n1, mx, p.dt);
#pragma unroll
    for (int wd = 0; wd < MASK_WORDS; ++wd) {
      if (wd < mask_words(p.steps)) p.masks[n1 * mask_words(p.steps) + wd] = mask[wd];
      if (mask[wd]) atomicOr((unsigned long long*)&p.flags[wd], (unsigned long long)mask[wd]);
    }
  }
}

// Per group its latest improvement at or before the stop step, which every wave finds by replaying the host loop's
// patience rule on the per-step "any group improved" flags (uniform, a few dozen scalar operations).  Reads and writes 16 bytes a
// group.  GROUPS of them a thread, whose loads are on their way at once; the step's factor comes from the table (it was a double
// division).  Four where that leaves every CU two workgroups, so that one replay serves 256 groups of a wave: 3.7 M groups
// 47 -> 24 us; one below, where the waves of a CU are few and four groups after the other take longer (a whole search of 0.3 M
// MXFP4 groups 51.4 us with four, 49.3 with one).
constexpr int64_t SELECT_FOUR_MIN_GROUPS = 1 << 19;
template <int WORDS, int GROUPS>
__global__ __launch_bounds__(256) void mse_select_kernel(const uint64_t* __restrict__ masks, int64_t n,
                                                         const uint64_t* __restrict__ flags, const float* __restrict__ factors,
                                                         int steps, int patience, int dt,
                                                         const void* __restrict__ min0,
                                                         const void* __restrict__ max0,
                                                         void* __restrict__ min_out, void* __restrict__ max_out) {
  __shared__ float factor[WORDS * 64];
  uint64_t any[WORDS], mask[GROUPS][WORDS];
  float mn[GROUPS], mx[GROUPS];
  const int64_t first = (int64_t)blockIdx.x * (256 * GROUPS) + threadIdx.x;
#pragma unroll
  for (int wd = 0; wd < WORDS; ++wd) any[wd] = flags[wd];
#pragma unroll
  for (int j = 0; j < GROUPS; ++j) {
    const int64_t i = first + 256 * j < n ? first + 256 * j : n - 1;
#pragma unroll
    for (int wd = 0; wd < WORDS; ++wd) mask[j][wd] = masks[i * WORDS + wd];
    mn[j] = load_rt(min0, i, dt);
    mx[j] = load_rt(max0, i, dt);
  }
  if (threadIdx.x < WORDS * 64) factor[threadIdx.x] = (int)threadIdx.x < steps ? factors[threadIdx.x] : 0.f;
  int no_improve = 0, last = -1;
#pragma unroll
  for (int wd = 0; wd < WORDS; ++wd) {
    const int end = steps - wd * 64 < 64 ? steps - wd * 64 : 64;
    for (int k = 0; k < end && last < 0; ++k) {
      no_improve = (any[wd] >> k) & 1ull ? 0 : no_improve + 1;
      if (no_improve >= patience) last = wd * 64 + k;
    }
  }
  if (last < 0) last = steps - 1;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < GROUPS; ++j) {
    const int64_t i = first + 256 * j;
    if (i >= n) break;
    int best = -1;
#pragma unroll
    for (int wd = WORDS - 1; wd >= 0; --wd) {
      const int upto = last - wd * 64;
      const uint64_t m = upto < 0 ? 0 : upto < 63 ? mask[j][wd] & ((2ull << upto) - 1ull) : mask[j][wd];
      if (best < 0 && m) best = wd * 64 + 63 - __clzll((long long)m);
    }
    // no recorded improvement (e.g. non-finite errors): the reference keeps the un-shrunk range
    const float pb = best < 0 ? 1.0f : factor[best];
    store_rt(min_out, i, best < 0 ? mn[j] : round_rt(product<LLMC_F16>(mn[j], pb), dt), dt);
    store_rt(max_out, i, best < 0 ? mx[j] : round_rt(product<LLMC_F16>(mx[j], pb), dt), dt);
  }
}

inline int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

// host-side round-to-nearest-even of a scalar to bf16 / f16
float round_host(float v, int dt) {
  if (dt == LLMC_BF16) {
    uint32_t u;
    memcpy(&u, &v, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    u &= 0xffff0000u;
    memcpy(&v, &u, 4);
    return v;
  }
  if (dt == LLMC_F16) return (float)(_Float16)v;
  return v;
}

struct Workspace {
  uint64_t* flags;
  float* factors;
  uint16_t* powtab;
  void* min0;
  void* max0;
  uint64_t* masks;
};

Workspace carve(void* ws, int64_t n) {
  char* c = (char*)ws;
  Workspace w;
  w.flags = (uint64_t*)c; c += 256;
  w.factors = (float*)c; c += MAX_STEPS * 4;
  w.powtab = (uint16_t*)c; c += 65536;
  w.min0 = c; c += align256(n * 4);
  w.max0 = c; c += align256(n * 4);
  w.masks = (uint64_t*)c;
  return w;
}

int finish(const MseParams& p, const Workspace& w, int64_t n, int patience, void* min_out, void* max_out,
           hipStream_t st) {
  LLMC_LAUNCH_STATUS();
  auto select = [&](auto kern, int groups) {
    hipLaunchKernelGGL(kern, dim3((unsigned)((n + 256 * groups - 1) / (256 * groups))), dim3(256), 0, st, w.masks, n, w.flags,
                       w.factors, p.steps, patience, p.dt, w.min0, w.max0, min_out, max_out);
  };
  const bool four = n >= SELECT_FOUR_MIN_GROUPS;
  if (mask_words(p.steps) == 1)
    four ? select(mse_select_kernel<1, 4>, 4) : select(mse_select_kernel<1, 1>, 1);
  else
    four ? select(mse_select_kernel<MASK_WORDS, 4>, 4) : select(mse_select_kernel<MASK_WORDS, 1>, 1);
  LLMC_LAUNCH_STATUS();
  return 0;
}

// `fast`: one of the 16-bit kernels follows, which read the power from a table unless it has a closed form
int setup(MseParams& p, Workspace& w, void* workspace, int64_t n, bool fast, hipStream_t st) {
  w = carve(workspace, n);
  p.min0 = w.min0;
  p.max0 = w.max0;
  p.masks = w.masks;
  p.flags = w.flags;
  p.factors = w.factors;
  const bool tab = fast && p.norm != 2.0f && p.norm != 3.0f && p.norm != 0.5f;
  if (tab) p.powtab = w.powtab;
  hipLaunchKernelGGL(mse_setup_kernel, dim3(tab ? 128 : 1), dim3(256), 0, st, w.flags, w.factors, p.steps, p.grid,
                     w.powtab, (int)tab, p.norm, p.dt);
  LLMC_LAUNCH_STATUS();
  return 0;
}

// long groups: in registers where they fit, else by re-reading them at every step
int launch_long(const MseParams& p, const GenericLayout& l, int64_t n, int64_t total, bool fast, hipStream_t st) {
  if (!fast) {
    hipLaunchKernelGGL(mse_generic_kernel, dim3((unsigned)n), dim3(256), 0, st, p, l);
    return 0;
  }
  return p.dt == LLMC_BF16 ? launch_rows_fast<LLMC_BF16>(p, l, n, (int)total, st)
                           : launch_rows_fast<LLMC_F16>(p, l, n, (int)total, st);
}

}  // namespace

extern "C" int64_t llmc_mse_workspace_bytes(int64_t n_groups) {
  return 256 + MAX_STEPS * 4 + 65536 + 2 * align256(n_groups * 4) + align256(n_groups * MASK_WORDS * 8);
}

static int check_common(int32_t dtype, int32_t fmt, int32_t num_bits, int32_t scale_mode, int32_t steps,
                        double grid, float norm, float expand, int32_t patience) {
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 2);
  LLMC_CHECK_ARG(fmt >= 0 && fmt <= 2, 100);
  LLMC_CHECK_ARG(fmt != LLMC_FMT_INT || (num_bits >= 2 && num_bits <= 8), 101);
  LLMC_CHECK_ARG(scale_mode == LLMC_SCALE_PLAIN || scale_mode == LLMC_SCALE_MXFP4, 102);
  LLMC_CHECK_ARG(steps >= 0 && steps <= MAX_STEPS, 103);
  LLMC_CHECK_ARG(grid > 0.0, 104);
  LLMC_CHECK_ARG(norm > 0.f && expand > 0.f && patience > 0, 105);
  return 0;
}

extern "C" int llmc_mse_observe_groups(const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                       int64_t group, int32_t fmt, int32_t num_bits, int32_t symmetric,
                                       int32_t scale_mode, int32_t steps, double grid, int32_t patience,
                                       float norm, float expand, void* min_out, void* max_out, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  LLMC_CHECK_ARG(x && R > 0 && K > 0, 1);
  int rc = check_common(dtype, fmt, num_bits, scale_mode, steps, grid, norm, expand, patience);
  if (rc) return rc;
  LLMC_CHECK_ARG(ldw >= K, 5);
  LLMC_CHECK_ARG(group > 0 && K % group == 0, 6);
  LLMC_CHECK_ARG(min_out && max_out, 16);
  const int64_t n = R * (K / group);
  LLMC_CHECK_ARG(workspace && (((uintptr_t)workspace) & 255) == 0 && workspace_bytes >= llmc_mse_workspace_bytes(n), 18);
  hipStream_t st = (hipStream_t)stream;
  MseParams p = {};
  p.x = x; p.dt = dtype; p.fmt = fmt; p.bits = fmt == LLMC_FMT_INT ? num_bits : (fmt == LLMC_FMT_FP8 ? 8 : 4);
  p.symmetric = symmetric; p.scale_mode = scale_mode; p.steps = steps; p.grid = grid; p.norm = round_host(norm, dtype); p.expand = expand;
  const int64_t L = group / 8;
  const bool team = dtype != LLMC_F32 && group % 8 == 0 && L <= 64 && (L & (L - 1)) == 0 && ldw % 8 == 0 &&
                    (((uintptr_t)x) & 15) == 0;
  const bool fast_team = team && (fmt != LLMC_FMT_FP4 || symmetric);
  const bool fast_rows = !team && rows_fast_ok(p, group);
  Workspace w;
  rc = setup(p, w, workspace, n, fast_team || fast_rows, st);
  if (rc) return rc;
  if (fast_team) {
    int lshift = 0;
    while ((1 << lshift) < L) ++lshift;
    rc = dtype == LLMC_BF16 ? launch_team_fast<LLMC_BF16>(p, n, (int)(K / group), (int)group, lshift, ldw, st)
                            : launch_team_fast<LLMC_F16>(p, n, (int)(K / group), (int)group, lshift, ldw, st);
  } else if (team) {
    const int64_t threads = n * L;
    hipLaunchKernelGGL(mse_team_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p, n,
                       (int)(K / group), (int)group, (int)L, ldw);
  } else {
    GenericLayout l = {};
    l.mode = 0; l.n0 = 1; l.G = group; l.s0 = 0; l.s1 = group; l.ldw = ldw;
    if (ldw != K) {
      // rows are not contiguous: one row at a time keeps the strided view valid
      LLMC_CHECK_ARG(group == K, 5);
      l.s1 = ldw;
    }
    rc = launch_long(p, l, n, group, fast_rows, st);
  }
  if (rc) return rc;
  return finish(p, w, n, patience, min_out, max_out, st);
}

static int observe_strided_impl(int err32, const void* x, int32_t dtype, int64_t n0, int64_t n1, int64_t group,
                                        int64_t stride0, int64_t stride1, int32_t fmt, int32_t num_bits,
                                        int32_t symmetric, int32_t scale_mode, int32_t steps, double grid,
                                        int32_t patience, float norm, float expand, void* min_out, void* max_out,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
  LLMC_CHECK_ARG(x && n0 > 0 && n1 > 0 && group > 0, 1);
  int rc = check_common(dtype, fmt, num_bits, scale_mode, steps, grid, norm, expand, patience);
  if (rc) return rc;
  LLMC_CHECK_ARG(min_out && max_out, 17);
  LLMC_CHECK_ARG(workspace && (((uintptr_t)workspace) & 255) == 0 && workspace_bytes >= llmc_mse_workspace_bytes(n1), 19);
  hipStream_t st = (hipStream_t)stream;
  MseParams p = {};
  p.x = x; p.dt = dtype; p.fmt = fmt; p.bits = fmt == LLMC_FMT_INT ? num_bits : (fmt == LLMC_FMT_FP8 ? 8 : 4);
  p.symmetric = symmetric; p.scale_mode = scale_mode; p.steps = steps; p.grid = grid;
  p.norm = err32 ? norm : round_host(norm, dtype); p.expand = expand; p.err32 = err32;
  Workspace w;
  rc = setup(p, w, workspace, n1, false, st);
  if (rc) return rc;
  GenericLayout l = {};
  l.mode = 0; l.n0 = n0; l.G = group; l.s0 = stride0; l.s1 = stride1;
  hipLaunchKernelGGL(mse_generic_kernel, dim3((unsigned)n1), dim3(256), 0, st, p, l);
  return finish(p, w, n1, patience, min_out, max_out, st);
}

extern "C" int llmc_mse_observe_strided(const void* x, int32_t dtype, int64_t n0, int64_t n1, int64_t group,
                                        int64_t stride0, int64_t stride1, int32_t fmt, int32_t num_bits,
                                        int32_t symmetric, int32_t scale_mode, int32_t steps, double grid,
                                        int32_t patience, float norm, float expand, void* min_out, void* max_out,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
  return observe_strided_impl(0, x, dtype, n0, n1, group, stride0, stride1, fmt, num_bits, symmetric, scale_mode, steps,
                              grid, patience, norm, expand, min_out, max_out, workspace, workspace_bytes, stream);
}

static int observe_blocks_impl(int err32, const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                       int32_t block_h, int32_t block_w, int32_t fmt, int32_t num_bits,
                                       int32_t symmetric, int32_t scale_mode, int32_t steps, double grid,
                                       int32_t patience, float norm, float expand, void* min_out, void* max_out,
                                       void* workspace, int64_t workspace_bytes, void* stream) {
  LLMC_CHECK_ARG(x && R > 0 && K > 0, 1);
  int rc = check_common(dtype, fmt, num_bits, scale_mode, steps, grid, norm, expand, patience);
  if (rc) return rc;
  LLMC_CHECK_ARG(block_h > 0 && block_w > 0, 6);
  const int nbr = (int)((R + block_h - 1) / block_h), nbc = (int)((K + block_w - 1) / block_w);
  const int64_t n = (int64_t)nbr * nbc;
  LLMC_CHECK_ARG(min_out && max_out, 17);
  LLMC_CHECK_ARG(workspace && (((uintptr_t)workspace) & 255) == 0 && workspace_bytes >= llmc_mse_workspace_bytes(n), 19);
  hipStream_t st = (hipStream_t)stream;
  MseParams p = {};
  p.x = x; p.dt = dtype; p.fmt = fmt; p.bits = fmt == LLMC_FMT_INT ? num_bits : (fmt == LLMC_FMT_FP8 ? 8 : 4);
  p.symmetric = symmetric; p.scale_mode = scale_mode; p.steps = steps; p.grid = grid;
  p.norm = err32 ? norm : round_host(norm, dtype); p.expand = expand; p.err32 = err32;
  Workspace w;
  const bool fast = rows_fast_ok(p, (int64_t)block_h * block_w);
  int bshift = -1;
  for (int k = 0; k < 15; ++k)
    if (block_w == 1 << k) bshift = k;
  rc = setup(p, w, workspace, n, fast, st);
  if (rc) return rc;
  GenericLayout l = {};
  l.mode = 1; l.bshift = bshift; l.R = (int)R; l.K = (int)K; l.bh = block_h; l.bw = block_w; l.nbc = nbc; l.ldw = ldw;
  rc = launch_long(p, l, n, (int64_t)block_h * block_w, fast, st);
  if (rc) return rc;
  return finish(p, w, n, patience, min_out, max_out, st);
}

extern "C" int llmc_mse_observe_blocks(const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                       int32_t block_h, int32_t block_w, int32_t fmt, int32_t num_bits,
                                       int32_t symmetric, int32_t scale_mode, int32_t steps, double grid,
                                       int32_t patience, float norm, float expand, void* min_out, void* max_out,
                                       void* workspace, int64_t workspace_bytes, void* stream) {
  return observe_blocks_impl(0, x, dtype, R, K, ldw, block_h, block_w, fmt, num_bits, symmetric, scale_mode, steps, grid,
                             patience, norm, expand, min_out, max_out, workspace, workspace_bytes, stream);
}

// ---- importance-weighted search (observers/imatrix.py) -------------------------------------------

namespace {

// partial[s][c] = sum over the s-th slice of the token rows of x[t][c]^2 (fp32, fixed order)
__global__ __launch_bounds__(256) void sumsq_partial_kernel(const void* __restrict__ x, int dt, int64_t T, int64_t K,
                                                            int64_t ldx, int slices, float* __restrict__ partial) {
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= K) return;
  const int s = blockIdx.y;
  const int64_t per = (T + slices - 1) / slices;
  const int64_t t0 = s * per, t1 = (t0 + per) < T ? t0 + per : T;
  float acc = 0.f;
  for (int64_t t = t0; t < t1; ++t) {
    const float v = load_rt(x, t * ldx + c, dt);
    acc += v * v;
  }
  partial[(int64_t)s * K + c] = acc;
}

__global__ __launch_bounds__(64) void sumsq_finish_kernel(const float* __restrict__ partial, int64_t K, int slices,
                                                          float* __restrict__ sum) {
  const int64_t c = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (c >= K) return;
  // the loads of 16 slices are issued together (one memory round trip per batch); the additions keep
  // the order s = 0, 1, 2, ...
  float acc = 0.f;
  int s = 0;
  for (; s + 16 <= slices; s += 16) {
    float v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = partial[(int64_t)(s + j) * K + c];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc += v[j];
  }
  for (; s < slices; ++s) acc += partial[(int64_t)s * K + c];
  sum[c] += acc;
}

constexpr int SUMSQ_SLICES = 64;

// 16-bit input with 16-byte aligned rows: a workgroup covers 256 columns of one token slice as 32 column
// groups (16-byte loads) x 8 token lanes, folds the token lanes through LDS and writes one partial row
__global__ __launch_bounds__(256) void sumsq_partial16_kernel(const uint16_t* __restrict__ x, int dt, int64_t T,
                                                              int64_t K, int64_t ldx, int slices,
                                                              float* __restrict__ partial) {
  __shared__ float red[8][256 + 8];
  const int cg = threadIdx.x & 31, tl = threadIdx.x >> 5;
  const int64_t c0 = (int64_t)blockIdx.x * 256 + cg * 8;
  const int s = blockIdx.y;
  const int64_t per = (T + slices - 1) / slices;
  const int64_t t0 = s * per, t1 = (t0 + per) < T ? t0 + per : T;
  float acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;
  if (c0 < K) {
    for (int64_t t = t0 + tl; t < t1; t += 8) {
      const uint4 v = *(const uint4*)(x + t * ldx + c0);
      float f[8];
      unpack8(v, dt, f);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += f[j] * f[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) red[tl][cg * 8 + j] = acc[j];
  __syncthreads();
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c < K) {
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 8; ++r) sum += red[r][threadIdx.x];
    partial[(int64_t)s * K + c] = sum;
  }
}

}  // namespace

extern "C" int64_t llmc_sumsq_workspace_bytes(int64_t K) { return align256(K * SUMSQ_SLICES * 4); }

// both entry points: partial sums of the token slices into `partial` ([slices, K] fp32), then sum += their total
static int sumsq_launch(const void* x, int32_t dtype, int64_t T, int64_t K, int64_t ldx, float* sum, float* partial,
                        hipStream_t st) {
  const int slices = T < SUMSQ_SLICES ? (int)T : SUMSQ_SLICES;
  const bool wide = dtype != LLMC_F32 && K % 8 == 0 && ldx % 8 == 0 && (((uintptr_t)x) & 15) == 0;
  if (wide)
    hipLaunchKernelGGL(sumsq_partial16_kernel, dim3((unsigned)((K + 255) / 256), (unsigned)slices), dim3(256), 0, st,
                       (const uint16_t*)x, dtype, T, K, ldx, slices, partial);
  else
    hipLaunchKernelGGL(sumsq_partial_kernel, dim3((unsigned)((K + 255) / 256), (unsigned)slices), dim3(256), 0, st, x,
                       dtype, T, K, ldx, slices, partial);
  LLMC_LAUNCH_STATUS();
  hipLaunchKernelGGL(sumsq_finish_kernel, dim3((unsigned)((K + 63) / 64)), dim3(64), 0, st,
                     (const float*)partial, K, slices, sum);
  LLMC_LAUNCH_STATUS();
  return 0;
}

extern "C" int llmc_sumsq_accumulate(const void* x, int32_t dtype, int64_t T, int64_t K, int64_t ldx, float* sum,
                                     void* workspace, int64_t workspace_bytes, void* stream) {
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 2);
  LLMC_CHECK_ARG(T >= 0 && K > 0 && ldx >= K, 3);
  if (T == 0) return 0;
  LLMC_CHECK_ARG(x != nullptr && sum != nullptr, 1);
  LLMC_CHECK_ARG(workspace && (((uintptr_t)workspace) & 255) == 0 && workspace_bytes >= llmc_sumsq_workspace_bytes(K), 7);
  return sumsq_launch(x, dtype, T, K, ldx, sum, (float*)workspace, (hipStream_t)stream);
}

// ---- the same accumulation for callers that cannot allocate ---------------------------------------
// The partial sums live in a device array of this library instead of a caller's workspace.  Every GPU
// that loads the library holds its own copy of the array (4 MiB) at its own address until the process
// ends; host code never uses the array's name as an address, only the pointer hipGetSymbolAddress
// returned for the device that is current.
constexpr int64_t SUMSQ_NOALLOC_MAX_K = LLMC_SUMSQ_NOALLOC_MAX_K;
static __device__ __align__(256) float scratch[SUMSQ_SLICES * SUMSQ_NOALLOC_MAX_K];

namespace {
constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
float* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// the address of `scratch` on the current device, looked up once per device
int scratch_for_current_device(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return 1000 + (int)e;
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return 2000;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return 1000 + (int)e;
    if (!p) return 2001;
    g_scratch_ptr[dev] = (float*)p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}
}  // namespace

extern "C" int llmc_sumsq_accumulate_noalloc(const void* x, int32_t dtype, int64_t T, int64_t K, int64_t ldx,
                                             float* sum, void* stream) {
  LLMC_CHECK_ARG(dtype >= 0 && dtype <= 2, 2);
  LLMC_CHECK_ARG(T >= 0 && ldx >= K, 3);
  // widths beyond the array's capacity are refused, never truncated
  LLMC_CHECK_ARG(K > 0 && K <= SUMSQ_NOALLOC_MAX_K, 4);
  if (T == 0) return 0;
  LLMC_CHECK_ARG(x != nullptr && sum != nullptr, 1);
  float* partial = nullptr;
  const int rc = scratch_for_current_device(&partial);
  if (rc) return rc;
  // every partial row that the finishing kernel reads is written by this call's first kernel, so the
  // contents that an earlier (possibly wider or longer) call left behind need no clearing
  return sumsq_launch(x, dtype, T, K, ldx, sum, partial, (hipStream_t)stream);
}

extern "C" int llmc_imatrix_observe_groups(const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                           int64_t group, int32_t fmt, int32_t num_bits, int32_t symmetric,
                                           int32_t scale_mode, int32_t steps, double grid, int32_t patience,
                                           float norm, float expand, const float* importance, void* min_out,
                                           void* max_out, void* workspace, int64_t workspace_bytes,
                                           void* stream) {
  LLMC_CHECK_ARG(x && R > 0 && K > 0, 1);
  // patience 0 = never stop early (imatrix.py:321-325)
  const int pat = patience > 0 ? patience : 0x7fffffff;
  int rc = check_common(dtype, fmt, num_bits, scale_mode, steps, grid, norm, expand, pat);
  if (rc) return rc;
  LLMC_CHECK_ARG(patience >= 0, 13);
  LLMC_CHECK_ARG(ldw >= K, 5);
  LLMC_CHECK_ARG(group > 0 && K % group == 0, 6);
  LLMC_CHECK_ARG(min_out && max_out, 17);
  const int64_t n = R * (K / group);
  LLMC_CHECK_ARG(workspace && (((uintptr_t)workspace) & 255) == 0 && workspace_bytes >= llmc_mse_workspace_bytes(n), 19);
  hipStream_t st = (hipStream_t)stream;
  MseParams p = {};
  p.x = x; p.dt = dtype; p.fmt = fmt; p.bits = fmt == LLMC_FMT_INT ? num_bits : (fmt == LLMC_FMT_FP8 ? 8 : 4);
  p.symmetric = symmetric; p.scale_mode = scale_mode; p.steps = steps; p.grid = grid; p.norm = norm; p.expand = expand;
  p.err32 = 1; p.imp = importance;
  Workspace w;
  rc = setup(p, w, workspace, n, false, st);
  if (rc) return rc;
  const int64_t L = group / 8;
  const bool team = dtype != LLMC_F32 && group % 8 == 0 && L <= 64 && (L & (L - 1)) == 0 && ldw % 8 == 0 &&
                    (((uintptr_t)x) & 15) == 0;
  if (team) {
    const int64_t threads = n * L;
    hipLaunchKernelGGL(mse_team_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, p, n,
                       (int)(K / group), (int)group, (int)L, ldw);
  } else {
    GenericLayout l = {};
    l.mode = 0; l.n0 = 1; l.G = group; l.s0 = 0; l.s1 = group; l.ldw = ldw; l.ng = K / group;
    if (ldw != K) {
      LLMC_CHECK_ARG(group == K, 5);
      l.s1 = ldw;
    }
    hipLaunchKernelGGL(mse_generic_kernel, dim3((unsigned)n), dim3(256), 0, st, p, l);
  }
  return finish(p, w, n, pat, min_out, max_out, st);
}

// the uniform fall-back of the importance-weighted observer on the other layouts (imatrix.py:141-245 route
// block-wise weights and non-weight observers to the same search without weights): fp32 error, patience 0 = never stop
extern "C" int llmc_imatrix_observe_strided(const void* x, int32_t dtype, int64_t n0, int64_t n1, int64_t group,
                                            int64_t stride0, int64_t stride1, int32_t fmt, int32_t num_bits,
                                            int32_t symmetric, int32_t scale_mode, int32_t steps, double grid,
                                            int32_t patience, float norm, float expand, void* min_out,
                                            void* max_out, void* workspace, int64_t workspace_bytes,
                                            void* stream) {
  LLMC_CHECK_ARG(patience >= 0, 14);
  return observe_strided_impl(1, x, dtype, n0, n1, group, stride0, stride1, fmt, num_bits, symmetric, scale_mode, steps,
                              grid, patience > 0 ? patience : 0x7fffffff, norm, expand, min_out, max_out, workspace,
                              workspace_bytes, stream);
}

extern "C" int llmc_imatrix_observe_blocks(const void* x, int32_t dtype, int64_t R, int64_t K, int64_t ldw,
                                           int32_t block_h, int32_t block_w, int32_t fmt, int32_t num_bits,
                                           int32_t symmetric, int32_t scale_mode, int32_t steps, double grid,
                                           int32_t patience, float norm, float expand, void* min_out,
                                           void* max_out, void* workspace, int64_t workspace_bytes, void* stream) {
  LLMC_CHECK_ARG(patience >= 0, 14);
  return observe_blocks_impl(1, x, dtype, R, K, ldw, block_h, block_w, fmt, num_bits, symmetric, scale_mode, steps, grid,
                             patience > 0 ? patience : 0x7fffffff, norm, expand, min_out, max_out, workspace,
                             workspace_bytes, stream);
}
