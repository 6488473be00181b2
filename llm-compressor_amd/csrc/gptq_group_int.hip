// Integer formats of the quantiser's group kernels (gptq_group.h): unrolled turns for 16-bit scales, loops for fp32 ones
// (models held in fp32).  4096 x 2048 weights, the whole loop (as one launch per block, before): bf16 scales 352 us unrolled
// (663), fp32 scales 437 as a loop (640), with zero points 436 (645); 16384 rows: 975 (1348), 1143 (1349), 1165 us (1364).
#include <type_traits>

#define LLMC_GPTQ_GROUP_KERNELS
#include "gptq_group.h"

GptqGroupKernels llmc_gptq_group_kernels_int(int sd, bool has_zp) {
  if (sd == LLMC_BF16)
    return has_zp ? unrolled_kernels<LLMC_FMT_INT, LLMC_BF16, true>() : unrolled_kernels<LLMC_FMT_INT, LLMC_BF16, false>();
  if (sd == LLMC_F16)
    return has_zp ? unrolled_kernels<LLMC_FMT_INT, LLMC_F16, true>() : unrolled_kernels<LLMC_FMT_INT, LLMC_F16, false>();
  return has_zp ? rolled_kernels<LLMC_FMT_INT, LLMC_F32, true>() : rolled_kernels<LLMC_FMT_INT, LLMC_F32, false>();
}
