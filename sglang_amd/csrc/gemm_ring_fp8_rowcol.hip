#include "gemm_ring_kernel.h"

namespace sglq {

void launch_ring_fp8_rowcol(GemmArgs& p, int config, int out_dtype, hipStream_t st) { launch_ring_kind<KIND_FP8_ROWCOL>(p, config, out_dtype, st); }

}  // namespace sglq
