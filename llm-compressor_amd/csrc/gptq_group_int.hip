// Integer formats of the quantiser's group kernels (gptq_group.h).
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
