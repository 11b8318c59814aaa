// Launches gemm_few_rows_kernel (gemm_few_rows.hip).
#pragma once
#include "gemm_device.h"

namespace sglq {
// p.ws: a plan for tiles of `rows` rows, 32 or 64, of at most max_tiles; p.N a multiple of 256, p.K of 128; codes to p.out [p.M][p.N / 2], scales to p.out_scales.
void launch_few_rows(GemmArgs& p, int max_tiles, int rows, int out_dtype, hipStream_t st);
}  // namespace sglq
