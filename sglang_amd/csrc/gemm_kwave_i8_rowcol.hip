#include "gemm_kwave_kernel.h"

namespace sglq {

void launch_kwave_i8_rowcol(GemmArgs& p, int config, int out_dtype, hipStream_t st) { launch_kwave_kind<KIND_I8_ROWCOL>(p, config, out_dtype, st); }

}  // namespace sglq
