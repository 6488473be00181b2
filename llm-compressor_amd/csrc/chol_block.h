// Workgroup-level pieces of the blocked Cholesky chain (512 threads = eight 64-wide waves, two per SIMD).
//
// factor_invert_64: Cholesky factor L of one 64 x 64 block and X = L^-1, left in LDS.  Columns stay unscaled (the L D L^T
// form: the update of column c by pivot column j is x[c] -= x[j] * (x_c[j] / d_j)), so no square root is on the chain, and a
// pivot that is not positive and finite is only recorded: what follows it is discarded by the caller.
//
// What bounds it is one wave's instruction issue: a vector instruction every 4.8 to 5.8 cycles (5.2 with a cross-lane operand),
// one that takes the result of the one before every 9.  A slab of 16 columns is therefore factored in four blocks of four:
// the four pivots of a block on the vector ALU, which touch only the block's own columns, and the rest of the slab by one
// matrix instruction for all four.  16 x 16 tiles lie in registers as v_mfma_f32_16x16x4_f32 holds its result: lane
// (g = lane / 16, r = lane % 16) has row r of the tile, columns 4 g .. 4 g + 3, so that block b's columns are what the row b
// of lanes holds, a row of the matrix per lane, and a pivot's multipliers are operands across lanes of that row
// (row_newbcast).  For the matrix instruction the four columns of the block are moved to the four rows of lanes (three lane
// swaps).  Waves 0 to 3 each keep the slab's diagonal tile -- the same arithmetic in each, so nothing crosses waves -- and
// one more tile that takes the same column operations: wave u > 0 the rows of tile row K + u, wave 0 rows of the identity,
// which end up as the transposed inverse of the unit-lower factor.  The tiles of the next slab are brought up to date in the
// registers that will factor them.
// 2750 cycles for the last slab, 3150 for the ones before it with their tiles' update, 14.9k for the block.  Pivot by pivot,
// one wave with all of a slab's rows and a cross-lane multiply-add per column: 3500 a slab, 17.3k the block.
//
// Everything of the inverse that can be formed by then, and the tiles behind the next slab, follow in the other waves,
// which have SIMDs of their own for it.  With X_kk = L_kk^-1 and W_k = -L[below, k] X_kk, the parts of X below the diagonal are
//   X_10 = X_11 W_0[1],  Z_0 = W_0[2..3] - L[2..3, 1] X_10,  X_2c = X_22 Z_c[2],  X_3c = X_33 (Z_c[3] + W_2[3] Z_c[2])
// (c = 0, 1 with Z_1 = W_1, and X_32 = X_33 W_2[3]), which needs one 16 x 16 product per wave and slab.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace cholblk {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int NB = 64;
constexpr int NT = 512;  // threads per workgroup
constexpr int LDD = 68;  // LDS row stride (floats) of a 64-wide block: 16-byte aligned rows, staggered banks
constexpr int LDP = 20;  // LDS row stride of a 16-wide tile
constexpr int LOW_ROWS = 48 + 32 + 16;

// 64 KB: with what a region's workgroup keeps beside it (chol_region.h), two workgroups fit a CU.
struct FactorScratch {
  float X[NB][LDD];          // the result: inverse of the factor, zeros above the diagonal
  float M[10][16][LDP];      // the block's tiles on and below the diagonal, row-major: tile(i, j)
  float V[LOW_ROWS][LDP];    // low(V, k, r)[t]: unscaled factored columns of slab k below its diagonal block (L = V D^-1/2)
  float T[LOW_ROWS][LDP];    // low(T, k, r)[t] = V / d: the unit-lower factor
  float W[LOW_ROWS][LDP];    // low(W, k, r)[c] = -(L[r, slab k] X_kk)[c]
  float Y[4][16][LDP];       // Y[k]: inverse of slab k's 16 x 16 unit-lower factor, row-major
  float Z[2][16][LDP];       // Z_0[2], Z_0[3]
  float Q[2][16][LDP];       // Z_c[3] + W_2[3] Z_c[2], c = 0, 1
  float rs[NB];              // 1 / L[r][r]
  int bad;                   // smallest column whose pivot was not positive and finite, NB if none
  int pad[3];
  __device__ float* tile(int i, int j) { return &M[i * (i + 1) / 2 + j][0][0]; }
  // row r of slab k: only the rows below the slab's diagonal block are kept, 48 + 32 + 16 of them
  __device__ static float* low(float (*m)[LDP], int k, int r) { return m[r - 16 + (k == 0 ? 0 : k == 1 ? 32 : 48)]; }
};

// ---- tiles in registers: v4f of row lane % 16, columns 4 (lane / 16) .. + 3 -------------------------------------------
__device__ __forceinline__ v4f tile_get(const float* t, int lane) {
  const float4 x = *(const float4*)(t + (lane & 15) * LDP + 4 * (lane >> 4));
  return v4f{x.x, x.y, x.z, x.w};
}
__device__ __forceinline__ void tile_put(v4f x, float* t, int lane) {
  *(float4*)(t + (lane & 15) * LDP + 4 * (lane >> 4)) = make_float4(x[0], x[1], x[2], x[3]);
}

// The pivots of block B of a slab: s (the diagonal tile) and y (the wave's other tile), columns 4 B .. 4 B + 3 of both,
// which the row B of lanes holds.  rd: the pivots' reciprocals, t: s times them (both in the row B of lanes).  One asm
// statement because the order is the point: what waits for a result is kept apart by what does not.  Wait states: a register
// is read across lanes 2 after it was written, a reciprocal 1.  Results of matrix instructions are older than that: the
// product with `one` reads the last of them where the compiler sees it and waits as long as it takes.
template <int B>
__device__ __forceinline__ void block_pivots(v4f& s, v4f& y, v4f& rd, v4f& t, float one) {
  float s0 = s[0] * one, s1 = s[1], s2 = s[2], s3 = s[3], y0 = B == 0 ? y[0] * one : y[0], y1 = y[1], y2 = y[2], y3 = y[3];
  float r0, r1, r2, r3, t0, t1, t2, t3;
#define LLMC_BC(lane) " row_newbcast:" lane " row_mask:%[rows] bank_mask:0xf\n\t"
#define LLMC_RCP(r, s, lane) "v_rcp_f32_dpp " r ", " s LLMC_BC(lane)
#define LLMC_SUB(x, xv, tv, lane) "v_fmac_f32_dpp " x ", -" tv ", " xv LLMC_BC(lane)
  asm volatile(
      "s_nop 1\n\t"
      LLMC_RCP("%[r0]", "%[s0]", "%[l0]")
      "s_nop 0\n\t"
      "v_mul_f32 %[t0], %[s0], %[r0]\n\t"
      "s_nop 1\n\t"
      LLMC_SUB("%[s1]", "%[s0]", "%[t0]", "%[l1]")
      LLMC_SUB("%[y1]", "%[y0]", "%[t0]", "%[l1]")
      LLMC_SUB("%[s2]", "%[s0]", "%[t0]", "%[l2]")
      LLMC_RCP("%[r1]", "%[s1]", "%[l1]")
      LLMC_SUB("%[y2]", "%[y0]", "%[t0]", "%[l2]")
      "v_mul_f32 %[t1], %[s1], %[r1]\n\t"
      LLMC_SUB("%[s3]", "%[s0]", "%[t0]", "%[l3]")
      LLMC_SUB("%[y3]", "%[y0]", "%[t0]", "%[l3]")
      LLMC_SUB("%[s2]", "%[s1]", "%[t1]", "%[l2]")
      LLMC_SUB("%[y2]", "%[y1]", "%[t1]", "%[l2]")
      LLMC_SUB("%[s3]", "%[s1]", "%[t1]", "%[l3]")
      LLMC_RCP("%[r2]", "%[s2]", "%[l2]")
      LLMC_SUB("%[y3]", "%[y1]", "%[t1]", "%[l3]")
      "v_mul_f32 %[t2], %[s2], %[r2]\n\t"
      "s_nop 1\n\t"
      LLMC_SUB("%[s3]", "%[s2]", "%[t2]", "%[l3]")
      LLMC_SUB("%[y3]", "%[y2]", "%[t2]", "%[l3]")
      "s_nop 0\n\t"
      LLMC_RCP("%[r3]", "%[s3]", "%[l3]")
      "s_nop 0\n\t"
      "v_mul_f32 %[t3], %[s3], %[r3]\n\t"
      "s_nop 1"
      : [s0] "+v"(s0), [s1] "+v"(s1), [s2] "+v"(s2), [s3] "+v"(s3), [y0] "+v"(y0), [y1] "+v"(y1), [y2] "+v"(y2),
        [y3] "+v"(y3), [r0] "=&v"(r0), [r1] "=&v"(r1), [r2] "=&v"(r2), [r3] "=&v"(r3), [t0] "=&v"(t0), [t1] "=&v"(t1),
        [t2] "=&v"(t2), [t3] "=&v"(t3)
      : [l0] "n"(4 * B), [l1] "n"(4 * B + 1), [l2] "n"(4 * B + 2), [l3] "n"(4 * B + 3), [rows] "n"(1 << B));
#undef LLMC_BC
#undef LLMC_RCP
#undef LLMC_SUB
  s = v4f{s0, s1, s2, s3};
  y = v4f{y0, y1, y2, y3};
  rd = v4f{r0, r1, r2, r3};
  t = v4f{t0, t1, t2, t3};
}

// the row B of lanes of x[0], x[1], x[2], x[3], as the rows of lanes of one register
template <int B>
__device__ __forceinline__ float to_rows(v4f x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[0]), __float_as_uint(x[1]), false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[2]), __float_as_uint(x[3]), false, false);
  const auto c = __builtin_amdgcn_permlane32_swap(a[B & 1], b[B & 1], false, false);
  return __uint_as_float(c[B >> 1]);
}

// Block B of a slab and what it takes off the blocks behind it.  `out` takes the block's columns of y: (y, rd) -> stores.
template <int B, typename Out>
__device__ __forceinline__ void slab_block(v4f& s, v4f& y, int lane, float one, Out out) {
  v4f rd, t;
  block_pivots<B>(s, y, rd, t, one);
  const v4f done = y;
  if constexpr (B < 3) {
    // zeros for what is finished: a row that is not finite must not reach the pivots before it
    const bool behind = (lane & 15) >= 4 * B + 4;
    const float ts = to_rows<B>(t), ss = to_rows<B>(s), by = to_rows<B>(y);
    const float a = behind ? -ts : 0.f, bs = behind ? ss : 0.f;
    y = __builtin_amdgcn_mfma_f32_16x16x4f32(a, by, y, 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // s is the last (see block_pivots)
    s = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bs, s, 0, 0, 0);
  }
  out(std::integral_constant<int, B>{}, done, rd);
}

// Slab K in wave u (0 .. 3 - K): s its diagonal tile, y tile (K + u, K), or rows of the identity for u = 0.
template <int K>
__device__ __forceinline__ void factor_slab(v4f s, v4f y, int u, int lane, FactorScratch& f) {
  const int r = lane & 15, g = lane >> 4;
  const int row = 16 * (K + u) + r;
  float one = 1.f;
  asm("" : "+s"(one));
  float* const at = u == 0 ? &f.Y[K][0][r] : f.low(f.V, K < 3 ? K : 0, row);
  auto out = [&](auto block, const v4f& y, const v4f& rd) {
    constexpr int B = decltype(block)::value;
    if (g != B) return;
    if (u == 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) at[(4 * B + v) * LDP] = y[v];
    } else if constexpr (K < 3) {
      *(float4*)(at + 4 * B) = make_float4(y[0], y[1], y[2], y[3]);
      *(float4*)(at + LOW_ROWS * LDP + 4 * B) = make_float4(y[0] * rd[0], y[1] * rd[1], y[2] * rd[2], y[3] * rd[3]);  // in T
    }
  };
  slab_block<0>(s, y, lane, one, out);
  slab_block<1>(s, y, lane, one, out);
  slab_block<2>(s, y, lane, one, out);
  slab_block<3>(s, y, lane, one, out);
  if (u != 0) return;
  // per row of the diagonal tile, in the lane that holds its pivot: 1/sqrt(d) (hardware estimate plus one Newton step) and
  // the pivot check.  A pivot that is zero, negative, infinite or NaN gives an estimate that is infinite, zero or NaN,
  // and the Newton step turns each of those into NaN.
  const bool mine = g == r >> 2;
  const int v = r & 3;
  const float d = v == 0 ? s[0] : (v == 1 ? s[1] : (v == 2 ? s[2] : s[3]));
  float rs = __builtin_amdgcn_rsqf(d);
  rs = rs * (1.5f - 0.5f * d * rs * rs);
  if (mine) f.rs[row] = rs;
  const unsigned long long failed = __ballot(mine && !(rs > 0.f && rs < 3.0e38f && d <= 3.0e38f));
  if (failed != 0ull && lane == 0 && f.bad == NB) f.bad = 16 * K + (__builtin_ctzll(failed) & 15);  // slabs run in ascending order
}

// tile (i, j) of the block less slab K's contribution
template <int K>
__device__ __forceinline__ v4f updated_tile(FactorScratch& f, int i, int j, int lane) {
  v4f acc = tile_get(f.tile(i, j), lane);
  const int r = lane & 15, g = lane >> 4;
  const float4 t = *(const float4*)(f.low(f.T, K, 16 * j + r) + 4 * g), v = *(const float4*)(f.low(f.V, K, 16 * i + r) + 4 * g);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-t.x, v.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-t.y, v.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-t.z, v.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-t.w, v.w, acc, 0, 0, 0);
  return acc;
}
template <int K>
__device__ __forceinline__ void update_tile(FactorScratch& f, int i, int j, int lane) {
  tile_put(updated_tile<K>(f, i, j, lane), f.tile(i, j), lane);
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

// `first`: tile (i, 0) of the block, called in waves 0 to 3 for i = 0 and i = their own number; the other tiles on and below
// the diagonal are in f.M when waves 4 to 7 return from beside() for the first time (or before); a barrier has passed since
// f was last read  ->  f.X = inverse of the block's lower Cholesky factor, exact zeros above the diagonal.  Every one of the
// 512 threads calls it.  Returns, in every thread, the smallest column whose pivot was not positive and finite (NB if none;
// the numbers computed after such a pivot are meaningless).  Ends with a barrier: f.X is readable by all on return.
// Waves 4 to 7 call beside() once while each of the four slabs is factored.
template <typename First, typename Beside>
__device__ __forceinline__ int factor_invert_64(FactorScratch& f, int tid, First first, Beside beside) {
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), r = tid & 63;
  const v4f identity = {(r & 15) == 4 * (r >> 4) ? 1.f : 0.f, (r & 15) == 4 * (r >> 4) + 1 ? 1.f : 0.f,
                        (r & 15) == 4 * (r >> 4) + 2 ? 1.f : 0.f, (r & 15) == 4 * (r >> 4) + 3 ? 1.f : 0.f};
  if (tid == 0) f.bad = NB;
  if (w < 4) {
    const v4f s = first(0);
    factor_slab<0>(s, w == 0 ? identity : first(w), w, r, f);
  } else {
    for (int i = tid - 256; i < NB * 16; i += NT - 256) {  // the tiles above the diagonal
      const int row = i >> 4, c4 = (i & 15) * 4;
      if ((c4 >> 4) > (row >> 4)) *(float4*)&f.X[row][c4] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    beside();
  }
  __syncthreads();
  if (w < 3) {
    const v4f s = updated_tile<0>(f, 1, 1, r);
    factor_slab<1>(s, w == 0 ? identity : updated_tile<0>(f, 1 + w, 1, r), w, r, f);
  } else if (w == 3) {
    update_tile<0>(f, 2, 2, r);
    update_tile<0>(f, 3, 2, r);
    update_tile<0>(f, 3, 3, r);
  } else {
    if (w == 7) {
#pragma unroll
      for (int i = 1; i < 4; ++i) product_tile<true>(f.low(f.T, 0, 16 * i), LDP, &f.Y[0][0][0], LDP, nullptr, 0, f.low(f.W, 0, 16 * i), LDP, r);
      diagonal_tile(f, 0, r);
    }
    beside();
  }
  __syncthreads();
  if (w < 2) {
    const v4f s = updated_tile<1>(f, 2, 2, r);
    factor_slab<2>(s, w == 0 ? identity : updated_tile<1>(f, 3, 2, r), w, r, f);
  } else if (w == 2) {
    update_tile<1>(f, 3, 3, r);
    product_tile<true>(f.low(f.T, 1, 32), LDP, &f.Y[1][0][0], LDP, nullptr, 0, f.low(f.W, 1, 32), LDP, r);
    product_tile<true>(f.low(f.T, 1, 48), LDP, &f.Y[1][0][0], LDP, nullptr, 0, f.low(f.W, 1, 48), LDP, r);
  } else if (w == 3) {
    product_tile<false>(&f.Y[1][0][0], LDP, f.low(f.W, 0, 16), LDP, nullptr, 0, &f.X[16][0], LDD, r, nullptr, &f.rs[16]);
    product_tile<true>(f.low(f.V, 1, 32), LDP, &f.X[16][0], LDD, f.low(f.W, 0, 32), LDP, &f.Z[0][0][0], LDP, r, &f.rs[16]);
    product_tile<true>(f.low(f.V, 1, 48), LDP, &f.X[16][0], LDD, f.low(f.W, 0, 48), LDP, &f.Z[1][0][0], LDP, r, &f.rs[16]);
  } else {
    if (w == 6) diagonal_tile(f, 1, r);
    beside();
  }
  __syncthreads();
  if (w == 0) {
    factor_slab<3>(updated_tile<2>(f, 3, 3, r), identity, 0, r, f);
  } else if (w == 1) {
    product_tile<false>(&f.Y[2][0][0], LDP, &f.Z[0][0][0], LDP, nullptr, 0, &f.X[32][0], LDD, r, nullptr, &f.rs[32]);
  } else if (w == 2) {
    product_tile<false>(&f.Y[2][0][0], LDP, f.low(f.W, 1, 32), LDP, nullptr, 0, &f.X[32][16], LDD, r, nullptr, &f.rs[32]);
    diagonal_tile(f, 2, r);
  } else if (w == 3) {
    product_tile<true>(f.low(f.T, 2, 48), LDP, &f.Y[2][0][0], LDP, nullptr, 0, f.low(f.W, 2, 48), LDP, r);
    product_tile<false>(f.low(f.W, 2, 48), LDP, &f.Z[0][0][0], LDP, &f.Z[1][0][0], LDP, &f.Q[0][0][0], LDP, r);
    product_tile<false>(f.low(f.W, 2, 48), LDP, f.low(f.W, 1, 32), LDP, f.low(f.W, 1, 48), LDP, &f.Q[1][0][0], LDP, r);
  } else {
    beside();
  }
  __syncthreads();
  // X_33 as its unscaled form and the row scale: its own tile is written at the same time
  if (w < 2) product_tile<false>(&f.Y[3][0][0], LDP, &f.Q[w][0][0], LDP, nullptr, 0, &f.X[48][16 * w], LDD, r, nullptr, &f.rs[48]);
  if (w == 2) product_tile<false>(&f.Y[3][0][0], LDP, f.low(f.W, 2, 48), LDP, nullptr, 0, &f.X[48][32], LDD, r, nullptr, &f.rs[48]);
  if (w == 3) diagonal_tile(f, 3, r);
  __syncthreads();
  return f.bad;
}

}  // namespace cholblk

// ---- 64-deep products on the matrix cores, one 16 x 16 tile per wave.  Tile layout of v_mfma_f32_16x16x4_f32: lane l
// holds column l % 16, rows 4 * (l / 16) + v.  Tile t of a 64 x 64 block: rows 16 (t / 4), columns 16 (t % 4).
namespace cholblk {

// 16 rows of 64 values as the matrix instruction takes them: the k index a lane group feeds into an instruction is free
// as long as both operands agree, so lane group g = lane / 16 takes k = 16 q + 4 g .. + 3 of row lane % 16 for the four
// instructions of chunk q and reads its 16 values as four 16-byte loads.
struct Operand64 {
  float4 v[4];
};
__device__ __forceinline__ Operand64 operand_load(const float* p, int64_t ld, int lane) {
  const float* src = p + (int64_t)(lane & 15) * ld + 4 * (lane >> 4);
  Operand64 o;
#pragma unroll
  for (int q = 0; q < 4; ++q) o.v[q] = *(const float4*)(src + 16 * q);
  return o;
}
// acc +/- X Y^T, over the first 16 * chunks indices
template <bool NEG>
__device__ __forceinline__ v4f tile_mm(v4f acc, const Operand64& x, const Operand64& y, int chunks = 4) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q >= chunks) break;
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
