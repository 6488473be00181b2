// Floating-point formats of the quantiser's group kernels (gptq_group.h): unrolled turns for what presets use (fp8 with
// 16-bit scales, fp4 with a global scale or with bf16 power-of-two scales), loops for the rest, which halve the code and
// the time to compile it.  4096 x 2048 weights, the whole loop (as one launch per block, before): fp8 with bf16 scales
// 350 us unrolled (702); with fp32 scales 438 as a loop (694), with zero points 471 (718); fp4 with f16 scales 454 (739).
// 16384 rows: 993 (1399), 1156 (1400), 1198 (1415), 1182 us (1432).
#include <type_traits>

#define LLMC_GPTQ_GROUP_KERNELS
#include "gptq_group.h"

GptqGroupKernels llmc_gptq_group_kernels_fp(int fmt, int sd, bool has_zp) {
  if (fmt == LLMC_FMT_FP8) {
    if (sd == LLMC_BF16)
      return has_zp ? rolled_kernels<LLMC_FMT_FP8, LLMC_BF16, true>() : unrolled_kernels<LLMC_FMT_FP8, LLMC_BF16, false>();
    if (sd == LLMC_F16)
      return has_zp ? rolled_kernels<LLMC_FMT_FP8, LLMC_F16, true>() : unrolled_kernels<LLMC_FMT_FP8, LLMC_F16, false>();
    return has_zp ? rolled_kernels<LLMC_FMT_FP8, LLMC_F32, true>() : rolled_kernels<LLMC_FMT_FP8, LLMC_F32, false>();
  }
  if (sd == LLMC_BF16)
    return has_zp ? rolled_kernels<LLMC_FMT_FP4, LLMC_BF16, true>() : unrolled_kernels<LLMC_FMT_FP4, LLMC_BF16, false>();
  if (sd == LLMC_F16)
    return has_zp ? rolled_kernels<LLMC_FMT_FP4, LLMC_F16, true>() : rolled_kernels<LLMC_FMT_FP4, LLMC_F16, false>();
  return has_zp ? rolled_kernels<LLMC_FMT_FP4, LLMC_F32, true>() : unrolled_kernels<LLMC_FMT_FP4, LLMC_F32, false>();
}
