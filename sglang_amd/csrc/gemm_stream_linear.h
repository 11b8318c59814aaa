// gemm_stream_quant_kernel and gemm_stream_tokenquant_kernel: the linear of up to eight rows in one launch, gemm_stream_kernel
// with the activation quantization folded in (groups of 128 to FP8; per token to FP8 or INT8).
//
// What bounds the two launches on so few rows is the first one: 2-3 us for a quantization of a few thousand values, which the
// GEMM's launch waits for.  In one launch every block of weight rows has to quantize the activations for itself, and what that
// costs is where it stands.  Here:
//   * the 16-bit activations are the first loads of the kernel, into registers: vector-memory operations retire in order, so
//     nothing waits for the weights behind them, which are on their way meanwhile (the former kernels had them travel through
//     the rings beside the weights, 2 KiB a K block whatever the rows, and read the rows once more for their maxima behind
//     the first weight copies);
//   * a wave holds exactly the K blocks that it multiplies, so codes are exchanged with nobody: one block barrier, for the rows' maxima
//     (per token), or none (groups).  A K block of a row lies on 16 lanes (8 for eight rows);
//     what 64 lanes hold in a register, K blocks times rows, is a unit;
//   * a unit is quantized while the copies of the step before it arrive, into one of two places in LDS in the operand layout;
//   * the rings carry weights only, two and four copies per K block and wave for 16 and 32 weight rows instead of five to eight; 29 and 54 KiB of LDS.
// Codes and scales come from the expressions of the quantization kernels, K is split over the waves and summed as in
// gemm_stream_kernel<KIND, 1, NIB>: the result is that of the two launches through that kernel bit for bit.
// Measured (graph-timed, weights rotated past the last-level cache; two launches / the former single kernels / here, us): block-FP8
// 1 x 2112 x 7168 9.6 / 8.6 / 7.0, 1 x 4096 x 4096 7.7 / 6.4 / 5.3, 1 x 10240 x 8192 20.6 / 20.3 / 16.9, 4 x 4096 x 4096 7.9 / 6.2 / 6.0, 8 x 14336 x 4096
// 15.4 / 14.3 / 13.9; per-token FP8 1 x 6144 x 4096 9.6 / 8.2 / 7.0, 1 x 28672 x 4096 25.0 / 24.1 / 21.3, 1 x 4096 x 14336 16.1 / 14.0 / 12.6, 4 x 4096 x
// 4096 7.9 / 7.7 / 5.7, 8 x 4096 x 4096 7.9 / 9.1 / 6.2; INT8 1 x 14336 x 4096 15.5 / 13.6 / 12.5, 4 x 8192 x 8192 17.1 / 16.5 / 14.4.  The GEMM alone, on quantized
// activations, takes 21.2 us on 1 x 28672 x 4096 and 12.3 on 1 x 14336 x 4096.
// Tried: all codes of a block formed before the K loop, shared by its waves (1 x 4096 x 4096 5.8 us, but 0.35 us for every 2048 activations:
// 4 x 4096 x 4096 7.9, 8 x 28672 x 4096 42); four K blocks of one row to a unit whatever the rows, quantized in one go (4 x 4096 x 4096 6.9).
#pragma once
#include "gemm_device.h"

namespace sglq {

// p.a: 16-bit activations [M, K], M <= 8, p.lda the row stride in bytes, K a multiple of 128; nib 1 or 2: 16 or 32 weight rows to a
// block; one function per kind, each in a translation unit of its own.
void launch_stream_fp8_block_linear(GemmArgs& p, int nib, int in_dtype, int out_dtype, hipStream_t st);
void launch_stream_fp8_token_linear(GemmArgs& p, int nib, int in_dtype, int out_dtype, hipStream_t st);
void launch_stream_i8_token_linear(GemmArgs& p, int nib, int in_dtype, int out_dtype, hipStream_t st);

}  // namespace sglq
