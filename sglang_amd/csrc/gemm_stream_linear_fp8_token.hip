#include "gemm_stream_linear_kernel.h"

namespace sglq {

void launch_stream_fp8_token_linear(GemmArgs& p, int nib, int in_dtype, int out_dtype, hipStream_t st) { launch_stream_linear<KIND_FP8_ROWCOL>(p, nib, in_dtype, out_dtype, st); }

}  // namespace sglq
