// The quantiser's column loop inside one group of column blocks (up to 512 columns): kernels and their parameters.
// Launched once per group by gptq.hip, instantiated in gptq_group_int.hip and gptq_group_fp.hip.
//
// What bounds it: rows are independent, but every column of a row depends on the one before it, so a wave works
// through 128 dependent steps per block.  A wave issues an independent vector instruction every 4.8 to 5.8 cycles and a
// dependent one every 9, and a SIMD completes one every 4 however many waves it holds.  Both kernels are therefore
// laid out for few instructions on that chain:
//   * a row belongs to a team of 16 or 8 lanes, each holding runs of 4 neighbouring columns in registers.  In every
//     turn each lane evaluates its own run with its own column constants.  Only the lane whose turn it is has final
//     values; a lane's later evaluations repeat its own, because the LDS copy of U holds zeros below the diagonal and
//     in the 4 x 4 diagonal blocks, so nothing is taken off a finished run.  Nothing is selected, stored or branched on
//     inside a turn; after the last turn of a run every lane holds its columns' values and errors;
//   * a turn's four errors reach the team as DPP operands (an immediate lane number, hence the unrolled turns), without
//     a pass through LDS;
//   * a division is three operations (quotient() below); a wave that meets a divisor or a value outside the range
//     where that gives the IEEE quotient repeats its block with plain divisions.
// Before block b is quantised, the group's earlier errors are taken off its columns on the matrix cores,
// W[:, b] - E U[:, b], as 16 x 16 tiles accumulated by v_mfma_f32_16x16x4_f32 in fp32.  In the left-looking form the same
// products bring in what the group owes to all earlier columns, P U[group, group]: E starts out as P in LDS, a block's own
// columns of it are multiplied ahead of the block before, and its errors are added to them.  As a pass over the pieces of P,
// a 512-wide product and a pass that formed D this took three launches more per group: without them 4096 x 4096
// 2441 -> 2181 us (a whole call), 4096 x 14336 19.7 -> 18.6 ms, 32 of 768 x 2048 5341 -> 4867 us.
//
// A workgroup is four waves that run the chain, one per SIMD, and four that prepare the next block meanwhile: its slice
// of U, its scales and the part of its tiles that does not wait for the current block.
//   16 lanes per row (16 rows per workgroup): the shortest chain, for weights that the chip takes in one pass.
//   A 4096-row group takes 48 us (as four block launches and three update launches: 124 us), 51 - 58 with P and D.
//   8 lanes per row (32 rows per workgroup): a turn has a quarter more instructions for twice the rows.  24576 rows:
//   210 us per group (before: 314 us), 236 with P and D.
// Both apply the same operations to every element in the same order, so they give the same bits.
#pragma once
#include "common.h"
#include "qformat.h"

constexpr int GB = 128;       // widest column block held on chip
constexpr int GROUP = 4;      // column blocks whose updates of the far columns are applied together
constexpr int Q_LDE = GROUP * GB;      // row stride of the scaled errors in memory

// One problem of a grouped call (llmc_gptq_quantize_grouped); the kernels pick theirs by a grid index and
// find its work buffers at a fixed stride behind those of problem 0.
struct GptqItem {
  const void* weight;
  const void* scale;
  const int8_t* zp;
  const float* gscale;
  const int32_t* g_idx;
  void* out;
};

struct GptqGroupParams {
  float* Wf;        // [rows up to a multiple of 128, ldw] fp32 work copy (permuted columns)
  int64_t ldw;
  int R;
  const float* U;   // inverse-Hessian upper factor
  int64_t ldu;
  int g0, gend, bs; // columns [g0, gend) in blocks of bs
  const void* scale;
  int scale_dt;
  const int8_t* zp;
  const float* gscale;
  const int32_t* g_idx;  // group of each (permuted) column, or NULL
  int64_t row_div, srow;
  int fmt, bits;
  int sd;           // dtype the dequantised value is formed in
  float* E;         // scaled errors of the group, negated, row stride Q_LDE; NULL with P or D
  float* loss_rows; // [R], written by the first group and added to by the others
  // grouped call: problem blockIdx.y takes scale / zp / gscale / g_idx from items and its Wf, U, E and
  // loss rows at these strides (in elements)
  const GptqItem* items;
  int64_t u_stride, w_stride, e_stride;
  // the left-looking form (gptq.hip), blocks of 128 columns: `pieces` matrices [.., Q_LDE] whose sum P times U[group, group]
  // the group's 512 columns take from the columns before them (0: nothing), and D (NULL: nobody reads it), the group's
  // columns of W minus the quantised ones over k_scale, [.., ldw] like Wf, with the rows' largest values so far and the
  // scales that follow from them
  const float* P;
  int pieces;
  int64_t piece_stride, p_stride;
  float* D;
  const float* k_scale;  // [K] per problem
  float *row_max, *row_scale;
  int64_t ks_stride, rows_stride;
};

typedef void (*GptqGroupKernel)(GptqGroupParams);
struct GptqGroupKernels {
  GptqGroupKernel few, many;  // 16 and 8 lanes per row
};
// by element format; fmt / sd as in GptqGroupParams
GptqGroupKernels llmc_gptq_group_kernels_int(int sd, bool has_zp);
GptqGroupKernels llmc_gptq_group_kernels_fp(int fmt, int sd, bool has_zp);

constexpr int QG = 4;                           // neighbouring columns per run
constexpr int Q_UHALF = GB / 2;
constexpr int Q_U = Q_UHALF * GB + Q_UHALF * Q_UHALF;  // LDS slice of U: rows 0..63 whole, rows 64..127 from column 64 on
constexpr int Q_D = GB / QG * 16;               // LDS column constants: four float4 per quad of columns
constexpr int Q_LDS_W = GB + 4;                 // LDS row stride of a block's values
constexpr int Q_LDS_E = GROUP * GB + 4;         // LDS row stride of the group's errors (and P)
constexpr int Q_THREADS = 512;
constexpr int q_rows(int team) { return 256 / team; }
constexpr int q_smem(int team, bool has_zp) {
  return (Q_U + Q_D + q_rows(team) * (2 * Q_LDS_W + Q_LDS_E)) * 4 + (has_zp ? q_rows(team) * Q_LDS_W : 0);
}

// the power of two that brings m >= 0 into [2^13, 2^14), the largest one for m = 0; 1 where m is not finite
constexpr int SCALE_MAX_EXP = 100;
__device__ __forceinline__ float scale_to_2_13(float m) {
  if (!(m <= 3.4028234e38f)) return 1.f;
  int e = 14 - SCALE_MAX_EXP;
  if (m > 0.f) (void)frexpf(m, &e);  // m in [2^(e-1), 2^e)
  e = 14 - e;
  return ldexpf(1.f, e < -SCALE_MAX_EXP ? -SCALE_MAX_EXP : (e > SCALE_MAX_EXP ? SCALE_MAX_EXP : e));
}

#ifdef LLMC_GPTQ_GROUP_KERNELS
namespace {

// The IEEE quotient x / s in three operations, from y = 1/s (hardware estimate, within an ulp, and one Newton step):
// q = RN(x y) is within 1.5 ulp of x / s, its residual x - q s is exact, and RN(q + residual * y) errs by no more than
// 1.5 * 2^-24 ulp (3 * 2^-24 where y is an ulp off) before its own rounding.  A quotient of two 24-bit numbers keeps
// 2^-25 ulp and multiples of that from every midpoint, so only numerators within a few such steps of one can go wrong;
// all 360 million of those up to 16 steps were tried, and every numerator of the 32 divisors whose y need not be the
// rounded reciprocal.  Two pairs fail, with the significands 0xfffffd and 0xffffff as divisors; those are refused.
// Refused divisors (also outside [2^-46, 2^46], where a quotient that matters could under- or overflow on the way) have
// a NaN reciprocal, and the caller falls back to plain divisions.  A numerator below 2^-100 has a subnormal residual, so
// its quotient can be an ulp off: as a value's it rounds to zero on every grid either way, and as an error's it is
// 2^-54 at most.  The residual's +0 turns a -0 quotient into +0, as adding a zero point of zero does.
__device__ __forceinline__ float quotient_reciprocal(const float s) {
  const float y0 = __builtin_amdgcn_rcpf(s), y = fmaf(fmaf(-s, y0, 1.0f), y0, y0);
  const bool ok = s >= 0x1p-46f && s <= 0x1p46f && (__float_as_uint(s) & 0x7ffffdu) != 0x7ffffdu;
  return ok ? y : __builtin_nanf("");
}
__device__ __forceinline__ float quotient(float x, float s, float y) {
  const float q = x * y;
  return fmaf(fmaf(-q, s, x), y, q);
}

template <int SD>
__device__ __forceinline__ float round_sd(float x) {
  if (SD == LLMC_BF16) return round16_finite<LLMC_BF16>(x);
  if (SD == LLMC_F16) return round16_finite<LLMC_F16>(x);
  return x;
}

// clamp and round a quotient onto the element grid (round_to_grid() with the conversion instructions)
template <int FMT, bool EXACT>
__device__ __forceinline__ float grid_value(float v, float qmin, float qmax) {
  v = EXACT ? fminf(fmaxf(v, qmin), qmax) : __builtin_amdgcn_fmed3f(v, qmin, qmax);
  if (FMT == LLMC_FMT_INT) return rintf(v);
  if (FMT == LLMC_FMT_FP8) return hw_e4m3_pair_decode(hw_e4m3_pair(v, v)).x;
  return hw_e2m1_pair_decode(hw_e2m1_pair(v, v)).x;
}

// a lane's run: 4 columns of one row, and everything about those columns that its evaluation needs
struct QRun {
  float w[QG], s[QG], y[QG], z[QG];    // values, scales, their reciprocals, zero points
  float dn[QG], dy[QG];                // minus U's diagonal and its reciprocals
  float u01, u02, u03, u12, u13, u23;  // the 4 x 4 diagonal block of U above its diagonal
};
struct QResult {
  float q[QG], e[QG];  // dequantised values and negated scaled errors
};
// sum of (w - q)^2 / d^2 over a run
__device__ __forceinline__ float run_loss(const QResult& o) {
  return fmaf(o.e[3], o.e[3], fmaf(o.e[2], o.e[2], fmaf(o.e[1], o.e[1], o.e[0] * o.e[0])));
}

// One run, start to finish inside a lane: column m is quantised, its scaled error err = (w - q) / d (kept negated, so that
// every update is one in-place multiply-add) is applied to
// the columns of the run behind it (one fused multiply-subtract per element; the reference rounds the outer product
// before it subtracts, the fused form keeps the product exact), and so on.
template <int FMT, int SD, bool HAS_ZP, bool EXACT>
__device__ __forceinline__ void gptq_run(const QRun& r, QResult& o, float qmin, float qmax) {
  float w1 = r.w[1], w2 = r.w[2], w3 = r.w[3];
  auto column = [&](float wv, int m) {
    float v = EXACT ? wv / r.s[m] + 0.0f : quotient(wv, r.s[m], r.y[m]);
    if (HAS_ZP) v = v + r.z[m];
    float dq = grid_value<FMT, EXACT>(v, qmin, qmax);
    if (HAS_ZP) dq = round_sd<SD>(dq - r.z[m]);
    o.q[m] = round_sd<SD>(dq * r.s[m]);
    const float x = __fsub_rn(wv, o.q[m]);
    o.e[m] = EXACT ? x / r.dn[m] : quotient(x, r.dn[m], r.dy[m]);
    return o.e[m];
  };
  const float e0 = column(r.w[0], 0);
  w1 = fmaf(e0, r.u01, w1);
  w2 = fmaf(e0, r.u02, w2);
  w3 = fmaf(e0, r.u03, w3);
  const float e1 = column(w1, 1);
  w2 = fmaf(e1, r.u12, w2);
  w3 = fmaf(e1, r.u13, w3);
  const float e2 = column(w2, 2);
  w3 = fmaf(e2, r.u23, w3);
  column(w3, 3);
}
static_assert(QG == 4, "gptq_run() is written out for runs of four columns");

// lane LI's value in every lane of the team: a row of 16 lanes (row_newbcast), or each half of it by its own
template <int TEAM, int LI>
__device__ __forceinline__ float team_value(float v) {
  const int x = __float_as_int(v);
  const int lo = __builtin_amdgcn_mov_dpp(x, 0x150 + LI, 0xf, 0xf, true);
  return __int_as_float(TEAM == 16 ? lo : __builtin_amdgcn_update_dpp(lo, x, 0x158 + (LI & 7), 0xf, 0xc, false));
}

// of a normal power of two up to 2^126: its exponent negated
__device__ __forceinline__ float reciprocal_of_power_of_2(float s) { return __uint_as_float(0x7f000000u - __float_as_uint(s)); }

__device__ __forceinline__ void add_row(float (&w)[QG], float e, const float4& u) {
  w[0] = fmaf(e, u.x, w[0]);
  w[1] = fmaf(e, u.y, w[1]);
  w[2] = fmaf(e, u.z, w[2]);
  w[3] = fmaf(e, u.w, w[3]);
}
// row i of the LDS slice of U at column c (c >= 64 where i >= 64)
__device__ __forceinline__ float4 u_row(const float* __restrict__ Us, int i, int c) {
  return *(const float4*)(i < Q_UHALF ? Us + i * GB + c : Us + Q_UHALF * GB + (i - Q_UHALF) * Q_UHALF + c - Q_UHALF);
}

// keeps the loads of one phase out of the phase before it (registers)
__device__ __forceinline__ void phase_end() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// the values are final here: without it their updates are put off, and the rows of U they take kept, to the end
__device__ __forceinline__ void settle(float (&w)[QG]) {
  asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
}

// Run J of lane t covers columns 4 TEAM J + 4 t .. + 3.
// Turn LI of run J, what it takes off the lanes' run J, and the turns after it.  What the turns of run J take off the later
// runs is applied one turn later (`ep`: the errors of the turn before), in the gaps of the evaluation's dependent chain.
// The rows of U are asked for before the evaluation; a turn is one scheduling region, which bounds the registers.
template <int TEAM, int J, int LI, int FMT, int SD, bool HAS_ZP>
__device__ __forceinline__ void gptq_turns(QRun& run, float (&w)[32 / TEAM][QG], QResult& o, float (&ep)[QG],
                                           const float* __restrict__ Us, int tl, float qmin, float qmax) {
  constexpr int NRUN = 32 / TEAM, SPAN = TEAM * QG;
  constexpr bool LAST = LI == TEAM - 1;
  float4 h[QG], g[QG][NRUN];
#pragma unroll
  for (int m = 0; m < QG; ++m) {
    if (!LAST) h[m] = u_row(Us, J * SPAN + LI * QG + m, J * SPAN + tl * QG);
    if (LI > 0) {
#pragma unroll
      for (int k = J + 1; k < NRUN; ++k) g[m][k] = u_row(Us, J * SPAN + (LI - 1) * QG + m, k * SPAN + tl * QG);
    }
  }
  gptq_run<FMT, SD, HAS_ZP, false>(run, o, qmin, qmax);
#pragma unroll
  for (int m = 0; m < QG; ++m) {
    if (LI > 0) {
#pragma unroll
      for (int k = J + 1; k < NRUN; ++k) add_row(w[k], ep[m], g[m][k]);
    }
    ep[m] = team_value<TEAM, LI>(o.e[m]);
    if (!LAST) add_row(run.w, ep[m], h[m]);
  }
  if (LAST) {
#pragma unroll
    for (int m = 0; m < QG; ++m)
#pragma unroll
      for (int k = J + 1; k < NRUN; ++k) add_row(w[k], ep[m], u_row(Us, J * SPAN + LI * QG + m, k * SPAN + tl * QG));
  }
#pragma unroll
  for (int k = J + 1; k < NRUN; ++k) settle(w[k]);
  phase_end();
  if constexpr (!LAST) gptq_turns<TEAM, J, LI + 1, FMT, SD, HAS_ZP>(run, w, o, ep, Us, tl, qmin, qmax);
}

// The turns of one run as a loop, operation for operation the same: formats without unrolled turns, and (EXACT) the rare
// way round with plain divisions.
template <int TEAM, int J, int FMT, int SD, bool HAS_ZP, bool EXACT>
__device__ __forceinline__ void gptq_turns_rolled(QRun& run, float (&w)[32 / TEAM][QG], QResult& o,
                                                  const float* __restrict__ Us, int tl, int count, float qmin, float qmax) {
  constexpr int NRUN = 32 / TEAM, SPAN = TEAM * QG;
#pragma unroll 1
  for (int li = 0; li < TEAM; ++li) {
    // columns at or past `count` hold w = 0, scale 1, d = 1 and zeros of U: nothing comes of their turns
    if (J * SPAN + li * QG >= count) break;
    gptq_run<FMT, SD, HAS_ZP, EXACT>(run, o, qmin, qmax);
    // a finished run meets zeros of U; the test keeps an error that is not finite away from it
    const bool open = tl > li;
#pragma unroll
    for (int m = 0; m < QG; ++m) {
      const float e = __shfl(o.e[m], li, TEAM);
      const int i = J * SPAN + li * QG + m;
      if (open) add_row(run.w, e, u_row(Us, i, J * SPAN + tl * QG));
#pragma unroll
      for (int k = J + 1; k < NRUN; ++k) add_row(w[k], e, u_row(Us, i, k * SPAN + tl * QG));
    }
  }
}

// base[row_off + off] with the base and the row offset uniform: a scalar address and one 32-bit lane offset (in elements;
// the offsets stay within 128 rows of at most 65536 values)
template <typename T>
__device__ __forceinline__ T load_at(const float* __restrict__ base, int64_t row_off, uint32_t off) {
  return *(const T*)((const char*)(base + row_off) + (off << 2));
}

// ---- the block's slice of U: entries above the 4 x 4 diagonal blocks, zeros elsewhere and past `count` --------------
// NQ quads per thread f = tid + n * nt.  Whole aligned blocks: fetch() issues the loads, put() stores them; others are
// copied by put() alone.
__device__ __forceinline__ void put_u(float* __restrict__ Us, int f, float4 v, int count) {
  const int i = f >> 5, c = (f & 31) * 4;
  const bool keep = c > (i & ~3) && i < count;
  v.x = keep && c + 0 < count ? v.x : 0.f;
  v.y = keep && c + 1 < count ? v.y : 0.f;
  v.z = keep && c + 2 < count ? v.z : 0.f;
  v.w = keep && c + 3 < count ? v.w : 0.f;
  if (i < Q_UHALF)
    *(float4*)&Us[i * GB + c] = v;
  else if (c >= Q_UHALF)
    *(float4*)&Us[Q_UHALF * GB + (i - Q_UHALF) * Q_UHALF + c - Q_UHALF] = v;
}
template <int NQ, int NT>
struct USlice {
  float4 v[NQ];
  __device__ __forceinline__ void fetch(const float* __restrict__ base, int64_t ldu, bool whole, int tid) {
    if (!whole) return;
#pragma unroll
    for (int n = 0; n < NQ; ++n)
      v[n] = load_at<float4>(base, n * (NT / 32) * ldu, (uint32_t)(tid >> 5) * (uint32_t)ldu + (tid & 31) * 4);
  }
  __device__ __forceinline__ void put(float* __restrict__ Us, const float* __restrict__ base, int64_t ldu, int count,
                                      bool whole, int tid) const {
    if (whole) {
#pragma unroll
      for (int n = 0; n < NQ; ++n) put_u(Us, tid + n * NT, v[n], GB);
      return;
    }
#pragma unroll 1
    for (int n = 0; n < NQ; ++n) {
      const int f = tid + n * NT, i = f >> 5, c = (f & 31) * 4;
      const float* src = base + (int64_t)(i < count ? i : count - 1) * ldu;
      put_u(Us, f, make_float4(src[c + 0 < count ? c + 0 : count - 1], src[c + 1 < count ? c + 1 : count - 1],
                               src[c + 2 < count ? c + 2 : count - 1], src[c + 3 < count ? c + 3 : count - 1]), count);
    }
  }
};

// column constants of a block, for thread i < 128 (column i): Ds[comp][quad] float4 with comp 0 = -d, 1 = -1/d,
// 2 = u01 u02 u03 u12, 3 = u13 u23
struct DColumn {
  float u[QG];  // U[i][4 (i/4) .. + 3]; only entries from the diagonal on are used
  __device__ __forceinline__ void fetch(const float* __restrict__ base, int64_t ldu, int count, int i) {
    const float* src = base + (int64_t)(i < count ? i : count - 1) * ldu;
#pragma unroll
    for (int k = 0; k < QG; ++k) {
      const int c = (i & ~3) + k;
      u[k] = src[c < count ? c : count - 1];
    }
  }
  __device__ __forceinline__ void put(float* __restrict__ Ds, int count, int i) const {
    const int quad = i >> 2, m = i & 3;
    float v[QG];
#pragma unroll
    for (int k = 0; k < QG; ++k) v[k] = i < count && (i & ~3) + k < count ? u[k] : 0.f;
    const float di = m == 0 ? v[0] : (m == 1 ? v[1] : (m == 2 ? v[2] : v[3])), d = i < count ? di : 1.f;
    float* q = Ds + quad * 4;
    constexpr int COMP = GB / QG * 4;
    q[m] = -d;
    q[COMP + m] = -quotient_reciprocal(d);
    if (m == 0) {
      q[2 * COMP + 0] = v[1];
      q[2 * COMP + 1] = v[2];
      q[2 * COMP + 2] = v[3];
    } else if (m == 1) {
      q[2 * COMP + 3] = v[2];
      q[3 * COMP + 0] = v[3];
    } else if (m == 2) {
      q[3 * COMP + 1] = v[3];
    }
  }
};
__device__ __forceinline__ void load_d(QRun& r, const float* __restrict__ Ds, int quad) {
  constexpr int COMP = GB / QG * 4;
  const float4 a = *(const float4*)(Ds + quad * 4), b = *(const float4*)(Ds + COMP + quad * 4);
  const float4 c = *(const float4*)(Ds + 2 * COMP + quad * 4), d = *(const float4*)(Ds + 3 * COMP + quad * 4);
  r.dn[0] = a.x; r.dn[1] = a.y; r.dn[2] = a.z; r.dn[3] = a.w;
  r.dy[0] = b.x; r.dy[1] = b.y; r.dy[2] = b.z; r.dy[3] = b.w;
  r.u01 = c.x; r.u02 = c.y; r.u03 = c.z; r.u12 = c.w; r.u13 = d.x; r.u23 = d.y;
}

template <int N>
__device__ __forceinline__ void load_scales(float (&s)[N], const void* p, int dt, int64_t base, const int (&gi)[N]) {
  if (dt == LLMC_BF16) {
#pragma unroll
    for (int e = 0; e < N; ++e) s[e] = load_as_f32<LLMC_BF16>(p, base + gi[e]);
  } else if (dt == LLMC_F16) {
#pragma unroll
    for (int e = 0; e < N; ++e) s[e] = load_as_f32<LLMC_F16>(p, base + gi[e]);
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) s[e] = load_as_f32<LLMC_F32>(p, base + gi[e]);
  }
}
// a value the compiler knows nothing about: what is computed from it is not kept in registers from one block to the next
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// ---- tiles of W[:, block] - E U[:, block] --------------------------------------------------------------------------
// A wave's NR x 2 tiles of 16 x 16: rows 16 t + .. of the workgroup, columns col0 / col1 (of the lane) of the block.
// The inner index runs over earlier blocks of the group, 64 at a time and never across a block's end; lane group
// q = lane / 16 contributes indices 16 q .. 16 q + 15 of a chunk, one per matrix instruction.
constexpr int KS = 64, KL = KS / 4;
struct BChunk {
  float b0[KL], b1[KL];
  __device__ __forceinline__ void fetch(const float* __restrict__ src, int64_t ldu, int len, int col0, int col1, int q) {
    if (len == KS) {
      const uint32_t o = (uint32_t)(KL * q) * (uint32_t)ldu;
#pragma unroll
      for (int j = 0; j < KL; ++j) {
        b0[j] = load_at<float>(src, j * ldu, o + (uint32_t)col0);
        b1[j] = load_at<float>(src, j * ldu, o + (uint32_t)col1);
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < KL; ++j) {
      const uint32_t o = (uint32_t)(KL * q + j < len ? KL * q + j : len - 1) * (uint32_t)ldu;
      b0[j] = load_at<float>(src, 0, o + (uint32_t)col0);
      b1[j] = load_at<float>(src, 0, o + (uint32_t)col1);
    }
  }
};
// The sums start from zero and the chain adds them to W, in one rounding: they are the size of a quantisation step, the
// weights several of them, and every instruction rounds a sum.
template <int NR>
struct Tiles {
  f32x4_t acc[NR][2];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int t = 0; t < NR; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t][0][i] = acc[t][1][i] = 0.f;
  }
  // E: the workgroup's rows at the chunk's first column
  __device__ __forceinline__ void multiply(const BChunk& b, const float* __restrict__ E, int lde, bool vec, int len, int c,
                                           int q, bool second_only = false) {
#pragma unroll
    for (int t = 0; t < NR; ++t) {
      const float* src = E + (t * 16 + c) * lde + KL * q;
      float a[KL];
      if (vec) {
#pragma unroll
        for (int j = 0; j < KL; j += 4) {
          const float4 v = *(const float4*)(src + j);
          a[j] = v.x; a[j + 1] = v.y; a[j + 2] = v.z; a[j + 3] = v.w;
        }
      } else {
#pragma unroll
        for (int j = 0; j < KL; ++j) a[j] = src[KL * q + j < len ? j : 0];
      }
      if (len < KS) {
#pragma unroll
        for (int j = 0; j < KL; ++j) a[j] = KL * q + j < len ? a[j] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < KL; ++j) {
        if (!second_only) acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b.b0[j], acc[t][0], 0, 0, 0);
        acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b.b1[j], acc[t][1], 0, 0, 0);
      }
    }
  }
  // inner indices 0 .. kc - 1 (whole blocks of bs)
  __device__ __forceinline__ void accumulate(const float* __restrict__ U, int64_t ldu, const float* __restrict__ E, int lde,
                                             int kc, int bs, int col0, int col1, int c, int q) {
    if (kc <= 0) return;
    BChunk cur, nxt;
    int k = 0, left = bs, len = left < KS ? left : KS;
    cur.fetch(U, ldu, len, col0, col1, q);
#pragma unroll 1
    while (true) {
      int kn = k + len, ln = left - len;
      if (ln == 0) ln = bs;
      const bool more = kn < kc;
      const int nlen = ln < KS ? ln : KS;
      if (more) nxt.fetch(U + (int64_t)kn * ldu, ldu, nlen, col0, col1, q);
      multiply(cur, E + k, lde, (k & 3) == 0 && len == KS, len, c, q);
      if (!more) break;
      cur = nxt;
      k = kn;
      left = ln;
      len = nlen;
    }
  }
};

// UNROLL: the turns unrolled (formats in common use) or as a loop
template <int TEAM, int FMT, int SD, bool HAS_ZP, bool UNROLL>
__global__ __launch_bounds__(Q_THREADS) void gptq_group_kernel(GptqGroupParams p) {
  constexpr int ROWS = q_rows(TEAM), NRUN = 32 / TEAM, SPAN = TEAM * QG;
  constexpr int NR = ROWS / 16;  // tile rows
  extern __shared__ __attribute__((aligned(16))) float qsmem[];
  float* const Us = qsmem;                       // slice of U of this block
  float* const Ds = Us + Q_U;                    // its column constants
  float* const Es = Ds + Q_D;                    // P, then P plus the errors of the finished blocks
  float* const Ws = Es + ROWS * Q_LDS_E;         // what the block's values owe to earlier columns, to be added to them
  float* const Ss = Ws + ROWS * Q_LDS_W;         // scales
  int8_t* const Zs = (int8_t*)(Ss + ROWS * Q_LDS_W);  // zero points (HAS_ZP only)
  if (p.items) {
    const GptqItem it = p.items[blockIdx.y];
    p.scale = it.scale; p.zp = it.zp; p.gscale = it.gscale; p.g_idx = it.g_idx;
    p.Wf += (int64_t)blockIdx.y * p.w_stride;
    p.U += (int64_t)blockIdx.y * p.u_stride;
    if (p.E) p.E += (int64_t)blockIdx.y * p.e_stride;
    p.loss_rows += (int64_t)blockIdx.y * p.R;
    p.P += (int64_t)blockIdx.y * p.p_stride;
    if (p.D) p.D += (int64_t)blockIdx.y * p.w_stride;
    p.k_scale += (int64_t)blockIdx.y * p.ks_stride;
    p.row_max += (int64_t)blockIdx.y * p.rows_stride;
    p.row_scale += (int64_t)blockIdx.y * p.rows_stride;
  }
  const int row0 = blockIdx.x * ROWS;
  const bool has_p = p.pieces > 0;
  // P, its pieces added in their order, by all threads: `half` of the workgroup's float4s to a role
  auto load_p = [&](int half) {
    constexpr int N = ROWS * GROUP * GB / 4 / Q_THREADS;  // per thread
    const int tid = opaque(threadIdx.x & 255);
    const float* src = p.P + (int64_t)row0 * Q_LDE + (int64_t)half * (N * 256 * 4);
    float4 v[N];
#pragma unroll
    for (int n = 0; n < N; ++n) v[n] = *(const float4*)(src + (tid + n * 256) * 4);
#pragma unroll 1
    for (int k = 1; k < p.pieces; ++k) {
      src += p.piece_stride;
      float4 x[N];
#pragma unroll
      for (int n = 0; n < N; ++n) x[n] = *(const float4*)(src + (tid + n * 256) * 4);
#pragma unroll
      for (int n = 0; n < N; ++n) {
        v[n].x += x[n].x; v[n].y += x[n].y; v[n].z += x[n].z; v[n].w += x[n].w;
      }
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int f = half * (N * 256) + tid + n * 256;
      *(float4*)&Es[(f >> 7) * Q_LDS_E + (f & 127) * 4] = v[n];
    }
  };
  const bool vec_u = (p.ldu & 3) == 0 && (p.bs & 3) == 0 && ((uintptr_t)p.U & 15) == 0;

  // Barriers, in the order in which both roles pass them: "ready" (a block's slice, scales and values are in LDS), "read"
  // (the chain has the scales and values in registers), and, unless it was the last block, "errors" (its errors are
  // in LDS, and the chain is done with the slice).
  if (threadIdx.x >= 256) {  // ---- helpers: whole waves
#pragma unroll 1
    for (int i2 = p.g0;;) {
      const int count = p.gend - i2 < p.bs ? p.gend - i2 : p.bs;
      const int kc = i2 - p.g0, last = kc - p.bs;  // the block before starts at column `last` of the group
      const int tid = opaque(threadIdx.x - 256), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
      const int tl = tid % TEAM, team = tid / TEAM, row = row0 + team;
      const bool live = row < p.R;
      const float* const base = p.U + (int64_t)i2 * p.ldu + i2;
      const bool whole = vec_u && count == GB;
      USlice<16, 256> u;
      u.fetch(base, p.ldu, whole, tid);
      DColumn d;
      if (tid < GB) d.fetch(base, p.ldu, count, tid);
      {
        // scales and zero points for the columns and the row of the chain's lane of the same number
        constexpr int N = NRUN * QG;
        const int64_t sbase = ((int64_t)(live ? row : p.R - 1) / p.row_div) * p.srow;
        int gi[N];
        float s[N], z[N];
#pragma unroll
        for (int e = 0; e < N; ++e) {
          const int c = (e / QG) * SPAN + tl * QG + (e % QG);
          gi[e] = p.g_idx ? p.g_idx[i2 + (c < count ? c : count - 1)] : 0;
        }
        load_scales(s, p.scale, p.scale_dt, sbase, gi);
#pragma unroll
        for (int e = 0; e < N; ++e) z[e] = HAS_ZP ? (float)p.zp[sbase + gi[e]] : 0.f;
        const float gs = p.gscale ? p.gscale[0] : 1.f;
#pragma unroll
        for (int J = 0; J < NRUN; ++J) {
#pragma unroll
          for (int m = 0; m < QG; ++m) {
            const int e = QG * J + m;
            if (p.gscale) s[e] = s[e] / gs;
            const bool in = live && J * SPAN + tl * QG + m < count;
            s[e] = in ? s[e] : 1.f;
            z[e] = in ? z[e] : 0.f;
          }
          const int o = team * Q_LDS_W + J * SPAN + tl * QG;
          *(float4*)&Ss[o] = make_float4(s[4 * J], s[4 * J + 1], s[4 * J + 2], s[4 * J + 3]);
          if (HAS_ZP) *(char4*)&Zs[o] = make_char4((int8_t)z[4 * J], (int8_t)z[4 * J + 1], (int8_t)z[4 * J + 2], (int8_t)z[4 * J + 3]);
        }
      }
      phase_end();
      if (has_p && kc == 0) {
        load_p(1);
        __syncthreads();  // P
      }
      if (kc > 0 || has_p) {
        const int c = lane & 15, q = lane >> 4;
        const int ct0 = wave * 16 + c, ct1 = ct0 + Q_UHALF;
        const int col0 = ct0 < count ? ct0 : count - 1, col1 = ct1 < count ? ct1 : count - 1;
        const float* const Uc = p.U + (int64_t)p.g0 * p.ldu + i2;
        Tiles<NR> tiles;
        tiles.clear();
        if (has_p) {  // the block's own columns of P; U's rows from 64 on are zero in the columns before them
          BChunk b;
          b.fetch(base, p.ldu, KS, col0, col1, q);
          tiles.multiply(b, Es + kc, Q_LDS_E, true, KS, c, q);
          b.fetch(base + (int64_t)KS * p.ldu, p.ldu, KS, col0, col1, q);
          tiles.multiply(b, Es + kc + KS, Q_LDS_E, true, KS, c, q, true);
        }
        tiles.accumulate(Uc, p.ldu, Es, Q_LDS_E, last, p.bs, col0, col1, c, q);
        phase_end();
        if (kc > 0) {
          // rows of U for the errors of the block before, in flight until they are there
          const int len0 = p.bs < KS ? p.bs : KS, len1 = p.bs - len0;
          BChunk b0, b1;
          b0.fetch(Uc + (int64_t)last * p.ldu, p.ldu, len0, col0, col1, q);
          if (len1 > 0) b1.fetch(Uc + (int64_t)(last + KS) * p.ldu, p.ldu, len1, col0, col1, q);
          __syncthreads();  // errors
          tiles.multiply(b0, Es + last, Q_LDS_E, (last & 3) == 0 && len0 == KS, len0, c, q);
          if (len1 > 0) tiles.multiply(b1, Es + last + KS, Q_LDS_E, (last & 3) == 0 && len1 == KS, len1, c, q);
        }
#pragma unroll
        for (int t = 0; t < NR; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            Ws[(t * 16 + 4 * q + i) * Q_LDS_W + ct0] = tiles.acc[t][0][i];
            Ws[(t * 16 + 4 * q + i) * Q_LDS_W + ct1] = tiles.acc[t][1][i];
          }
      }
      u.put(Us, base, p.ldu, count, whole, tid);
      if (tid < GB) d.put(Ds, count, tid);
      __syncthreads();  // ready
      __syncthreads();  // read
      i2 += count;
      if (i2 >= p.gend) return;
    }
  }

  // ---- the chain
  const QFormat f = make_qformat(FMT, p.bits);   // the format is a compile-time constant here
  const bool vec_w = (p.bs & 3) == 0;
  float loss = 0.f, dmax = 0.f;
  if (has_p) {
    load_p(0);
    __syncthreads();  // P
  }
#pragma unroll 1
  for (int i1 = p.g0; i1 < p.gend; i1 += p.bs) {
    const int count = p.gend - i1 < p.bs ? p.gend - i1 : p.bs;
    const int kc = i1 - p.g0;
    const bool more = i1 + count < p.gend;
    const int tid = opaque(threadIdx.x), tl = tid % TEAM, team = tid / TEAM, row = row0 + team;
    const bool live = row < p.R;
    float* const wrow = p.Wf + (int64_t)row * p.ldw;
    float* const erow = p.E + (int64_t)row * Q_LDE;
    float w[NRUN][QG], s[NRUN][QG], z[NRUN][QG];
    auto load_w = [&]() {  // as they are in memory
#pragma unroll
      for (int J = 0; J < NRUN; ++J) {
        const int c = J * SPAN + tl * QG;
        float4 v;
        if (vec_w)
          v = *(const float4*)&wrow[i1 + (c < count ? c : 0)];
        else
          v = make_float4(wrow[i1 + (c < count ? c : 0)], wrow[i1 + (c + 1 < count ? c + 1 : 0)],
                          wrow[i1 + (c + 2 < count ? c + 2 : 0)], wrow[i1 + (c + 3 < count ? c + 3 : 0)]);
        w[J][0] = v.x; w[J][1] = v.y; w[J][2] = v.z; w[J][3] = v.w;
      }
    };
    auto add_sums = [&]() {
#pragma unroll
      for (int J = 0; J < NRUN; ++J) {
        const int c = J * SPAN + tl * QG;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (kc > 0 || has_p) v = *(const float4*)&Ws[team * Q_LDS_W + c];
        w[J][0] = live && c + 0 < count ? w[J][0] + v.x : 0.f;
        w[J][1] = live && c + 1 < count ? w[J][1] + v.y : 0.f;
        w[J][2] = live && c + 2 < count ? w[J][2] + v.z : 0.f;
        w[J][3] = live && c + 3 < count ? w[J][3] + v.w : 0.f;
      }
    };
    load_w();
    __syncthreads();  // ready
    add_sums();
#pragma unroll
    for (int J = 0; J < NRUN; ++J) {
      const int o = team * Q_LDS_W + J * SPAN + tl * QG;
      const float4 a = *(const float4*)&Ss[o];
      const char4 b = HAS_ZP ? *(const char4*)&Zs[o] : make_char4(0, 0, 0, 0);
      s[J][0] = a.x; s[J][1] = a.y; s[J][2] = a.z; s[J][3] = a.w;
      z[J][0] = b.x; z[J][1] = b.y; z[J][2] = b.z; z[J][3] = b.w;
    }
    __syncthreads();  // read
    __builtin_amdgcn_s_setprio(3);  // the helper on the same SIMD takes what this wave leaves

    QResult o[NRUN];
#pragma unroll
    for (int J = 0; J < NRUN; ++J)
#pragma unroll
      for (int m = 0; m < QG; ++m) o[J].q[m] = o[J].e[m] = 0.f;
    bool bad = false;
    auto run_step = [&](auto tag, auto exact_tag) {
      constexpr int J = decltype(tag)::value;
      constexpr bool EXACT = decltype(exact_tag)::value;
      if (J * SPAN >= count) return;  // uniform
      QRun r;
      load_d(r, Ds, J * TEAM + tl);
#pragma unroll
      for (int m = 0; m < QG; ++m) {
        r.w[m] = w[J][m];
        r.s[m] = s[J][m];
        r.z[m] = z[J][m];
        r.y[m] = quotient_reciprocal(r.s[m]);
        bad = bad | (r.y[m] != r.y[m]);
      }
      if constexpr (UNROLL && !EXACT) {
        float ep[QG];
        gptq_turns<TEAM, J, 0, FMT, SD, HAS_ZP>(r, w, o[J], ep, Us, tl, f.qmin, f.qmax);
      } else {
        gptq_turns_rolled<TEAM, J, FMT, SD, HAS_ZP, EXACT>(r, w, o[J], Us, tl, count, f.qmin, f.qmax);
      }
    };
    auto all_runs = [&](auto exact_tag) {
      run_step(std::integral_constant<int, 0>{}, exact_tag);
      run_step(std::integral_constant<int, 1>{}, exact_tag);
      if constexpr (NRUN > 2) {
        run_step(std::integral_constant<int, 2>{}, exact_tag);
        run_step(std::integral_constant<int, 3>{}, exact_tag);
      }
      static_assert(NRUN == 2 || NRUN == 4, "one step per run of a lane");
    };
    all_runs(std::false_type{});
    float total = 0.f;
#pragma unroll
    for (int J = 0; J < NRUN; ++J) total += run_loss(o[J]);
    if (__any(bad || !(total < 0x1p60f))) {  // every quotient stayed below 2^128 then, or its NaN is in the total
      load_w();
      add_sums();
      all_runs(std::true_type{});
    }
    __builtin_amdgcn_s_setprio(0);
    if (more) {
#pragma unroll
      for (int J = 0; J < NRUN; ++J) {
        const int c = J * SPAN + tl * QG;
        if (vec_w && c + QG <= count) {
          float4* const at = (float4*)&Es[team * Q_LDS_E + kc + c];
          float4 v = make_float4(o[J].e[0], o[J].e[1], o[J].e[2], o[J].e[3]);
          if (has_p) {
            const float4 x = *at;
            v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
          }
          *at = v;
        } else {
#pragma unroll
          for (int m = 0; m < QG; ++m)
            if (c + m < count) Es[team * Q_LDS_E + kc + c + m] = o[J].e[m];
        }
      }
      __syncthreads();  // errors
    }
    // the row's loss in an order that does not depend on the team: lane t adds up the runs of 4 columns number t, t + 8,
    // t + 16, t + 24 of every block
#pragma unroll
    for (int J = 0; J < NRUN; ++J) {
      const float part = run_loss(o[J]);
      if (TEAM == 8) {
        loss += part;
      } else {
        loss += __shfl(part, tl & 7, 16);
        loss += __shfl(part, 8 + (tl & 7), 16);
      }
    }
    if (live) {
#pragma unroll
      for (int J = 0; J < NRUN; ++J) {
        const int c = J * SPAN + tl * QG;
        if (p.D) {  // (in whole blocks) the weights as they came are still in Wf
          const float4 w0 = *(const float4*)&wrow[i1 + c], ks = *(const float4*)&p.k_scale[i1 + c];
          float4 d = make_float4(w0.x - o[J].q[0], w0.y - o[J].q[1], w0.z - o[J].q[2], w0.w - o[J].q[3]);
          d.x *= reciprocal_of_power_of_2(ks.x); d.y *= reciprocal_of_power_of_2(ks.y);
          d.z *= reciprocal_of_power_of_2(ks.z); d.w *= reciprocal_of_power_of_2(ks.w);
          dmax = fmaxf(dmax, fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fmaxf(fabsf(d.z), fabsf(d.w))));
          *(float4*)&p.D[(int64_t)row * p.ldw + i1 + c] = d;
        }
        if (vec_w && c + QG <= count) {
          *(float4*)&wrow[i1 + c] = make_float4(o[J].q[0], o[J].q[1], o[J].q[2], o[J].q[3]);
          if (p.E) *(float4*)&erow[kc + c] = make_float4(o[J].e[0], o[J].e[1], o[J].e[2], o[J].e[3]);
        } else {
#pragma unroll
          for (int m = 0; m < QG; ++m)
            if (c + m < count) {
              wrow[i1 + c + m] = o[J].q[m];
              if (p.E) erow[kc + c + m] = o[J].e[m];
            }
        }
      }
    }
  }
  loss += __shfl_xor(loss, 1, 8);
  loss += __shfl_xor(loss, 2, 8);
  loss += __shfl_xor(loss, 4, 8);
  const int row = row0 + (int)threadIdx.x / TEAM;
  if (row < p.R && threadIdx.x % TEAM == 0) p.loss_rows[row] = (p.g0 == 0 ? 0.f : p.loss_rows[row]) + loss * 0.5f;
  if (p.D) {
#pragma unroll
    for (int k = 1; k < TEAM; k *= 2) dmax = fmaxf(dmax, __shfl_xor(dmax, k, TEAM));
    if (row < p.R && threadIdx.x % TEAM == 0) {
      if (p.g0 > 0) dmax = fmaxf(dmax, p.row_max[row]);
      p.row_max[row] = dmax;
      p.row_scale[row] = scale_to_2_13(dmax);
    }
  }
}

template <int FMT, int SD, bool HAS_ZP>
GptqGroupKernels unrolled_kernels() {
  return {gptq_group_kernel<16, FMT, SD, HAS_ZP, true>, gptq_group_kernel<8, FMT, SD, HAS_ZP, true>};
}
template <int FMT, int SD, bool HAS_ZP>
GptqGroupKernels rolled_kernels() {
  return {gptq_group_kernel<16, FMT, SD, HAS_ZP, false>, gptq_group_kernel<8, FMT, SD, HAS_ZP, false>};
}

}  // namespace
#endif
