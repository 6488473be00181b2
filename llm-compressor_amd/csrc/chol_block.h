// Workgroup-level pieces of the blocked Cholesky chain (512 threads = eight 64-wide waves, two per SIMD).
//
// factor_invert_64: Cholesky factor L of one 64 x 64 block and X = L^-1, left in LDS.
//
// The block lives in LDS; a column slab of 16 is factored by one wave.  What bounds it is that wave's issue: 64 pivots,
// one after the other, a vector instruction every 5.5 cycles and a dependent one every 9.  So the slab loop holds what
// the chain needs and nothing else:
//   * every row of 16 lanes keeps its own copy of the slab's diagonal rows (`b`, lane i = row i, 16 columns in
//     registers), so that a pivot's multipliers are operands of the updates themselves (v_fmac_f32_dpp with
//     row_newbcast: lane c of the own row of lanes); with v_readlane into scalars each took an instruction of its own
//     and a wait;
//   * a second set of registers (`a`) takes the same column operations: 48 lanes hold the rows below the diagonal block,
//     the first 16 lanes hold rows of the identity, which end up as the transposed inverse of the unit-lower factor --
//     no separate inversion;
//   * the columns stay unscaled (the L D L^T form): the update of column c by pivot column j is
//     x[c] -= x[j] * (b_c[j] / d_j), and no square root sits on the chain;
//   * a pivot that is not positive and finite is only recorded (one ballot per slab): what follows it is
//     discarded by the caller, so no fix-up sits on the chain either.
// Between two slabs the next slab's columns are updated on v_mfma_f32_16x16x4_f32 (one 16 x 16 tile per wave); the
// columns after it, and everything of the inverse that can be formed by then, follow in the other waves while the next
// slab is factored.  With X_kk = L_kk^-1 and W_k = -L[below, k] X_kk, the parts of X below the diagonal are
//   X_10 = X_11 W_0[1],  Z_0 = W_0[2..3] - L[2..3, 1] X_10,  X_2c = X_22 Z_c[2],  X_3c = X_33 (Z_c[3] + W_2[3] Z_c[2])
// with Z_1 = W_1[2..3] for column c = 1, and X_32 = X_33 W_2[3]: one product with X_33 is left after the last slab.
// About 6 us in all (with scalar multipliers, a vector-unit update and the inverse after each slab: 7.8 us).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cholblk {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int NB = 64;
constexpr int NT = 512;  // threads per workgroup
constexpr int LDD = 68;  // LDS row stride (floats) of a 64-wide block: 16-byte aligned rows, staggered banks
constexpr int LDP = 20;  // LDS row stride of a 16-wide slab
constexpr int LDA = 52;  // ... of a column of the 48 x 48 block behind the first slab
constexpr int LOW_ROWS = 48 + 32 + 16;

// 63 KB: with what a region's workgroup keeps beside it (chol_region.h), two workgroups fit a CU.
struct FactorScratch {
  float X[NB][LDD];          // the result: inverse of the factor, zeros above the diagonal
  float AT[NB - 16][LDA];    // the block, column-major: at(c, r) = A[r][c], columns and rows from 16 on
  float P[NB][LDP];          // the current slab's columns, row-major
  float V[LOW_ROWS][LDP];    // low(V, k, r)[t]: unscaled factored columns of slab k below its diagonal block (L = V D^-1/2)
  float T[LOW_ROWS][LDP];    // low(T, k, r)[t] = V / d: the unit-lower factor
  float W[LOW_ROWS][LDP];    // low(W, k, r)[c] = -(L[r, slab k] X_kk)[c]
  float Y[4][16][LDP];       // Y[k]: inverse of slab k's 16 x 16 unit-lower factor, row-major
  float Z[2][16][LDP];       // Z_0[2], Z_0[3]
  float rs[NB];              // 1 / L[r][r]
  int bad;                   // smallest column whose pivot was not positive and finite, NB if none
  int pad[3];
  __device__ float* at(int c, int r) { return &AT[c - 16][r - 16]; }
  // row r of slab k: only the rows below the slab's diagonal block are kept, 48 + 32 + 16 of them
  __device__ static float* low(float (*m)[LDP], int k, int r) { return m[r - 16 + (k == 0 ? 0 : k == 1 ? 32 : 48)]; }
  // Q_c = Z_c[3] + W_2[3] Z_c[2], c = 0, 1: in rows of P that the last slab does not use
  __device__ float* q(int c) { return P[16 * c]; }
};

// v in lane LI of every row of 16 lanes, for the whole row
template <int LI>
__device__ __forceinline__ float row_lane(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + LI, 0xf, 0xf, true));
}
// x[c] -= x_j * (lane c's t), c = J + 1 .. 15, in ascending order.  Written out in assembly because the compiler does
// not fold a broadcast with two uses into its multiply-adds.  A vector register may be read across lanes two
// wait states after it was written: hence the wait before the first (t) and, where the caller reads x[J + 1] across
// lanes (PIVOT), behind it.
template <int J, bool PIVOT, int C = J + 1>
__device__ __forceinline__ void eliminate(float (&x)[16], float xj, float t) {
  if constexpr (C < 16) {
    if constexpr (C == J + 1 && PIVOT)
      asm volatile("s_nop 1\n\tv_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\ts_nop 1"
                   : "+v"(x[C]) : "v"(t), "v"(xj), "n"(C));
    else if constexpr (C == J + 1)
      asm volatile("s_nop 1\n\tv_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                   : "+v"(x[C]) : "v"(t), "v"(xj), "n"(C));
    else
      asm volatile("v_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                   : "+v"(x[C]) : "v"(t), "v"(xj), "n"(C));
    eliminate<J, PIVOT, C + 1>(x, xj, t);
  }
}

template <int J>
__device__ __forceinline__ void pivots(float (&b)[16], float (&a)[16], float (&rd)[16], float& myd, int i) {
  if constexpr (J < 16) {
    rd[J] = __builtin_amdgcn_rcpf(row_lane<J>(b[J]));
    myd = i == J ? b[J] : myd;
    const float t = b[J] * rd[J];
    eliminate<J, true>(b, b[J], t);
    eliminate<J, false>(a, a[J], t);
    pivots<J + 1>(b, a, rd, myd, i);
  }
}

// Slab K, in one wave.
template <int K>
__device__ __forceinline__ void factor_slab(int lane, FactorScratch& s) {
  const int i = lane & 15, g = lane >> 4;
  const int row = 16 * (K + g) + i;         // g = 0: row of the diagonal block (and identity row i); g > 0: a row below
  const bool below = g > 0 && K + g < 4;
  float b[16], a[16], rd[16], myd = 1.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 x = *(const float4*)&s.P[16 * K + i][4 * q];
    b[4 * q] = x.x; b[4 * q + 1] = x.y; b[4 * q + 2] = x.z; b[4 * q + 3] = x.w;
    float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
    if (below) y = *(const float4*)&s.P[row][4 * q];
    a[4 * q] = y.x; a[4 * q + 1] = y.y; a[4 * q + 2] = y.z; a[4 * q + 3] = y.w;
  }
  if (g == 0) {
#pragma unroll
    for (int c = 0; c < 16; ++c) a[c] = c == i ? 1.f : 0.f;
  }
  pivots<0>(b, a, rd, myd, i);
  if (K < 3 && below) {
    constexpr int KK = K < 3 ? K : 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      *(float4*)(s.low(s.V, KK, row) + 4 * q) = make_float4(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
      *(float4*)(s.low(s.T, KK, row) + 4 * q) = make_float4(a[4 * q] * rd[4 * q], a[4 * q + 1] * rd[4 * q + 1],
                                                   a[4 * q + 2] * rd[4 * q + 2], a[4 * q + 3] * rd[4 * q + 3]);
    }
  }
  if (g == 0) {
#pragma unroll
    for (int c = 0; c < 16; ++c) s.Y[K][c][i] = a[c];
  }
  // per row of the diagonal block: 1/sqrt(d) (hardware estimate plus one Newton step) and the pivot check.  A
  // pivot that is zero, negative, infinite or NaN gives an estimate that is infinite, zero or NaN, and the
  // Newton step turns each of those into NaN.
  float rs = __builtin_amdgcn_rsqf(myd);
  rs = rs * (1.5f - 0.5f * myd * rs * rs);
  if (g == 0) s.rs[row] = rs;
  const unsigned long long failed = __ballot(g == 0 && !(rs > 0.f && rs < 3.0e38f && myd <= 3.0e38f));
  if (failed != 0ull && lane == 0 && s.bad == NB) s.bad = 16 * K + __builtin_ctzll(failed);  // slabs run in ascending order
}

// acc - A B^T over 16 inner indices, A[i][k] at A + i * LDP + k, B[c][k] at B + c * LDP + k
__device__ __forceinline__ v4f tile16_nt(v4f acc, const float* A, const float* B, int lane) {
  const int i = lane & 15, g = lane >> 4;
  const float4 av = *(const float4*)(A + i * LDP + 4 * g), bv = *(const float4*)(B + i * LDP + 4 * g);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-av.x, bv.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-av.y, bv.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-av.z, bv.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-av.w, bv.w, acc, 0, 0, 0);
  return acc;
}
// tile (ti, tj) of the block, less slab K's contribution: into P (the next slab's columns) or back into AT
template <int K>
__device__ __forceinline__ void update_tile(FactorScratch& s, int ti, int tj, bool to_panel, int lane) {
  const int c = lane & 15, g = lane >> 4;
  float* const at = s.at(16 * tj + c, 16 * ti + 4 * g);
  const float4 x = *(const float4*)at;
  v4f acc = {x.x, x.y, x.z, x.w};
  acc = tile16_nt(acc, s.low(s.V, K, 16 * ti), s.low(s.T, K, 16 * tj), lane);
  if (to_panel) {
#pragma unroll
    for (int v = 0; v < 4; ++v) s.P[16 * ti + 4 * g + v][c] = acc[v];
  } else {
    *(float4*)at = make_float4(acc[0], acc[1], acc[2], acc[3]);
  }
}
// 16 x 16 tile A B (+ C) into `out` (row stride ldo); A's columns scaled by ascale, its rows by rscale, negated with NEG
template <bool NEG>
__device__ __forceinline__ void product_tile(const float* A, int lda, const float* B, int ldb, const float* C, int ldc,
                                             float* out, int ldo, int lane, const float* ascale = nullptr,
                                             const float* rscale = nullptr) {
  const int c = lane & 15, g = lane >> 4;
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  if (C) {
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = C[(4 * g + v) * ldc + c];
  }
  const float rsc = rscale ? rscale[c] : 1.f;
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    float av = A[c * lda + 4 * kk + g];
    if (ascale) av *= ascale[4 * kk + g];
    if (rscale) av *= rsc;
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(NEG ? -av : av, B[(4 * kk + g) * ldb + c], acc, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) out[(4 * g + v) * ldo + c] = acc[v];
}
// X_kk = Y_k with its rows scaled by 1/L[r][r]
__device__ __forceinline__ void diagonal_tile(FactorScratch& s, int k, int lane) {
  const int r = lane >> 2, q = lane & 3;
  const float4 y = *(const float4*)&s.Y[k][r][4 * q];
  const float f = s.rs[16 * k + r];
  *(float4*)&s.X[16 * k + r][16 * k + 4 * q] = make_float4(y.x * f, y.y * f, y.z * f, y.w * f);
}

// the caller's share: row r of the block, columns 8 w .. 8 w + 7, as the 512 threads (w = tid / 64, r = tid % 64) hold it
__device__ __forceinline__ void factor_block_put(FactorScratch& s, float4 d0, float4 d1, int w, int r) {
  if (w < 2) {
    *(float4*)&s.P[r][8 * w] = d0;
    *(float4*)&s.P[r][8 * w + 4] = d1;
    return;
  }
  if (r < 16) return;  // above the diagonal
  float* const at = s.at(8 * w, r);
  at[0 * LDA] = d0.x; at[1 * LDA] = d0.y; at[2 * LDA] = d0.z; at[3 * LDA] = d0.w;
  at[4 * LDA] = d1.x; at[5 * LDA] = d1.y; at[6 * LDA] = d1.z; at[7 * LDA] = d1.w;
}

// factor_block_put() has been called by every thread of the 512 (its lower triangle incl. the diagonal is used); no
// barrier is needed in between  ->  s.X = inverse of the block's lower Cholesky factor, exact zeros above the
// diagonal.  Every one of the 512 threads calls it.  Returns, in every thread, the smallest column whose pivot was not
// positive and finite (NB if none; the numbers computed after such a pivot are meaningless).  Ends with a
// barrier: s.X is readable by all on return.  Waves 4 to 7 call beside() once while each of the four slabs is factored (1.5
// us each, in which they have at most one tile to form).
template <typename Beside>
__device__ __forceinline__ int factor_invert_64(FactorScratch& s, int tid, Beside beside) {
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), r = tid & 63;
  if (tid == 0) s.bad = NB;
  __syncthreads();

  if (w == 0) {
    factor_slab<0>(r, s);
  } else {
    for (int i = tid - 64; i < NB * 16; i += NT - 64) {  // the tiles above the diagonal
      const int row = i >> 4, c4 = (i & 15) * 4;
      if ((c4 >> 4) > (row >> 4)) *(float4*)&s.X[row][c4] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  if (w >= 4) beside();
  __syncthreads();
  if (w < 3) update_tile<0>(s, 1 + w, 1, true, r);
  if (w == 3) diagonal_tile(s, 0, r);
  __syncthreads();
  if (w == 0) factor_slab<1>(r, s);
  if (w == 1) update_tile<0>(s, 2, 2, false, r);
  if (w == 2) update_tile<0>(s, 3, 2, false, r);
  if (w == 3) update_tile<0>(s, 3, 3, false, r);
  if (w >= 4 && w < 7)
    product_tile<true>(s.low(s.T, 0, 16 * (w - 3)), LDP, &s.Y[0][0][0], LDP, nullptr, 0, s.low(s.W, 0, 16 * (w - 3)), LDP, r);
  if (w >= 4) beside();
  __syncthreads();
  if (w < 2) update_tile<1>(s, 2 + w, 2, true, r);
  if (w == 2) diagonal_tile(s, 1, r);
  __syncthreads();
  if (w == 0) factor_slab<2>(r, s);
  if (w == 1) update_tile<1>(s, 3, 3, false, r);
  if (w == 2 || w == 3) product_tile<true>(s.low(s.T, 1, 16 * w), LDP, &s.Y[1][0][0], LDP, nullptr, 0, s.low(s.W, 1, 16 * w), LDP, r);
  if (w == 4) product_tile<false>(&s.X[16][16], LDD, s.low(s.W, 0, 16), LDP, nullptr, 0, &s.X[16][0], LDD, r);
  if (w >= 4) beside();
  __syncthreads();
  if (w == 0) update_tile<2>(s, 3, 3, true, r);
  if (w == 1) diagonal_tile(s, 2, r);
  if (w == 2 || w == 3)
    product_tile<true>(s.low(s.V, 1, 16 * w), LDP, &s.X[16][0], LDD, s.low(s.W, 0, 16 * w), LDP, &s.Z[w - 2][0][0], LDP, r, &s.rs[16]);
  if (w == 4) product_tile<true>(s.low(s.T, 2, 48), LDP, &s.Y[2][0][0], LDP, nullptr, 0, s.low(s.W, 2, 48), LDP, r);
  __syncthreads();
  if (w == 0) factor_slab<3>(r, s);
  if (w == 1) product_tile<false>(&s.X[32][32], LDD, &s.Z[0][0][0], LDP, nullptr, 0, &s.X[32][0], LDD, r);
  if (w == 2) product_tile<false>(&s.X[32][32], LDD, s.low(s.W, 1, 32), LDP, nullptr, 0, &s.X[32][16], LDD, r);
  if (w == 3) product_tile<false>(s.low(s.W, 2, 48), LDP, &s.Z[0][0][0], LDP, &s.Z[1][0][0], LDP, s.q(0), LDP, r);
  if (w == 4) product_tile<false>(s.low(s.W, 2, 48), LDP, s.low(s.W, 1, 32), LDP, s.low(s.W, 1, 48), LDP, s.q(1), LDP, r);
  if (w >= 4) beside();
  __syncthreads();
  // X_33 as its unscaled form and the row scale: its own tile is written at the same time
  if (w < 2) product_tile<false>(&s.Y[3][0][0], LDP, s.q(w), LDP, nullptr, 0, &s.X[48][16 * w], LDD, r, nullptr, &s.rs[48]);
  if (w == 2) product_tile<false>(&s.Y[3][0][0], LDP, s.low(s.W, 2, 48), LDP, nullptr, 0, &s.X[48][32], LDD, r, nullptr, &s.rs[48]);
  if (w == 3) diagonal_tile(s, 3, r);
  __syncthreads();
  return s.bad;
}

}  // namespace cholblk

// ---- 64-deep products on the matrix cores, one 16 x 16 tile per wave.  Tile layout of v_mfma_f32_16x16x4_f32: lane l
// holds column l % 16, rows 4 * (l / 16) + v.  Tile t of a 64 x 64 block: rows 16 (t / 4), columns 16 (t % 4).
namespace cholblk {

// 16 rows of 64 values as the matrix instruction takes them: the k index a lane group feeds into an instruction is free
// as long as both operands agree, so lane group g = lane / 16 takes k = 16 g .. 16 g + 15 of row lane % 16 and reads
// its 16 values as four 16-byte loads.
struct Operand64 {
  float4 v[4];
};
__device__ __forceinline__ Operand64 operand_load(const float* p, int64_t ld, int lane) {
  const float* src = p + (int64_t)(lane & 15) * ld + 16 * (lane >> 4);
  Operand64 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o.v[q] = *(const float4*)(src + 4 * q);
  return o;
}
// acc +/- X Y^T
template <bool NEG>
__device__ __forceinline__ v4f tile_mm(v4f acc, const Operand64& x, const Operand64& y) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 a = x.v[q], b = y.v[q];
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(NEG ? -a.x : a.x, b.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(NEG ? -a.y : a.y, b.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(NEG ? -a.z : a.z, b.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(NEG ? -a.w : a.w, b.w, acc, 0, 0, 0);
  }
  return acc;
}
__device__ __forceinline__ v4f tile_load(const float* p, int64_t ld, int t, int lane) {
  const float* src = p + (int64_t)(16 * (t >> 2) + 4 * (lane >> 4)) * ld + 16 * (t & 3) + (lane & 15);
  return v4f{src[0], src[ld], src[2 * ld], src[3 * ld]};
}
__device__ __forceinline__ void tile_store(v4f acc, float* p, int64_t ld, int t, int lane) {
  float* dst = p + (int64_t)(16 * (t >> 2) + 4 * (lane >> 4)) * ld + 16 * (t & 3) + (lane & 15);
#pragma unroll
  for (int v = 0; v < 4; ++v) dst[v * ld] = acc[v];
}

}  // namespace cholblk
