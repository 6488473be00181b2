// Internal fp32 GEMM on the matrix cores (v_mfma_f32_32x32x2_f32), used for the
// chain's triangular inverse and the updates of the GPTQ and SparseGPT loops; B^T and lower triangles for llmc_sgemm.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct GemmF32 {
  // C[M,N] = alpha * A' * B' + beta * C,   all row-major
  //   trans_b = 0: B' = B,  B stored [Kc,N];   trans_b = 1: B' = B^T, B stored [N,Kc]
  //   trans_a = 0: A' = A,  A stored [M,Kc];   trans_a = 1: A' = A^T, A stored [Kc,M] (only with
  //   trans_b = 0 and without the a_lower_tri hint)
  const float* A;
  int64_t lda;
  const float* B;
  int64_t ldb;
  float* C;
  int64_t ldc;
  int M, N, Kc;
  float alpha, beta;
  int trans_b;
  int trans_a;
  // structure hints (tile-granular; operands must hold exact zeros where the structure says so)
  int c_lower;      // only tiles that touch the lower triangle of C are computed
  int a_lower_tri;  // A[m,k] = 0 for k > m : contraction stops at the tile's last row
  int b_lower_tri;  // B'[k,n] = 0 for k < n : contraction starts at the tile's first column
  int b_upper_tri;  // B'[k,n] = 0 for k > n : contraction stops at the tile's last column (the split kernels; others may
                    // multiply the zeros)
  // batching over blockIdx.z
  int batch;
  int64_t stride_a, stride_b, stride_c;
  // contraction length of the last block of the batch when it differs from Kc (a contraction cut into
  // `batch` pieces whose last one is shorter); 0 = Kc like the others
  int kc_last;
  // second batch level (independent problems, each with `batch` blocks): blockIdx.z = b + batch * b2;
  // 0 or 1 = none
  int batch2;
  int64_t stride2_a, stride2_b, stride2_c;
  // llmc_gemm_x2 only: A and B hold their elements split into two f16 terms already (split2.h)
  int split;
  // llmc_gemm_x2 only, powers of two: C = alpha * diag(row_scale)^-1 (diag(row_scale) A) (diag(k_scale) B), one k_scale
  // per index of the contraction (of the whole one when it is cut into pieces); strides per problem of batch2
  const float* row_scale;
  const float* k_scale;
  int64_t stride2_rs, stride2_ks;
};

// enqueue on `st`; returns 0 or 1000 + hipError_t
int llmc_gemm_f32(const GemmF32& g, hipStream_t st);

// The same product on the 16-bit matrix cores (every operand split into three bf16 planes, six partial
// products; see gemm_x3.hip): taken when the shape is a whole number of 64-wide tiles and long enough.
// Returns -1 when the product is left to the fp32 matrix instruction.
int llmc_gemm_x3(const GemmF32& g, hipStream_t st);
// 0 = never use the split product, 1 = whenever it applies (default)
void llmc_gemm_x3_set_mode(int mode);

// The product of operands whose range is known, split into two f16 terms (gemm_x2.hip): |A| and |B| (scaled, where scales
// are given) at most 2^15, at least one element of a row that matters near 2^13.  A B^T of operands that are split, A B with scales; takes
// what llmc_gemm_x2_fits.
bool llmc_gemm_x2_fits(const GemmF32& g);
int llmc_gemm_x2(const GemmF32& g, hipStream_t st);
