#include "gemm_ring_kernel.h"

namespace sglq {

void launch_ring_fp8_block_grouped(GemmArgs& p, int config, int out_dtype, hipStream_t st) {
  if (out_dtype == SGLQ_BF16) launch_ring_grouped_config<KIND_FP8_BLOCK, SGLQ_BF16>(p, config, st);
  else launch_ring_grouped_config<KIND_FP8_BLOCK, SGLQ_FP16>(p, config, st);
}

}  // namespace sglq
