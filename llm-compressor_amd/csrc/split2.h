// An fp32 value as two f16 terms (gemm_x2.hip), eight at a time: what a thread puts into LDS, and what a matrix that is split
// ahead of its products holds in the place of eight neighbouring elements -- their first terms, then their second ones.
#pragma once
#include "common.h"
#include "qformat.h"

// (x s, y t) -> the packed f16 pairs of the two planes; s and t are powers of two, so the remainder x s - a0 is exact in one
// fused operation that takes a0 as it is (v_fma_mix_f32; also for s = 1, if the compiler does not see that it is one)
__device__ __forceinline__ void split2(float x, float y, float s, float t, uint32_t& p0, uint32_t& p1) {
  p0 = pack16<LLMC_F16>(x * s, y * t);
  p1 = pack16<LLMC_F16>(__builtin_fmaf(x, s, -f16_bits_to_f32((uint16_t)p0)),
                        __builtin_fmaf(y, t, -f16_bits_to_f32((uint16_t)(p0 >> 16))));
}

__device__ __forceinline__ void split2_unscaled(float x, float y, float one, uint32_t& p0, uint32_t& p1) {
  p0 = pack16<LLMC_F16>(x, y);
  p1 = pack16<LLMC_F16>(__builtin_fmaf(x, one, -f16_bits_to_f32((uint16_t)p0)),
                        __builtin_fmaf(y, one, -f16_bits_to_f32((uint16_t)(p0 >> 16))));
}
