// gemm_kwave_kernel: the GEMM for 17 to some two thousand rows with small tiles, K split over the waves of a block.
//
// What bounds gemm_ring_kernel on such tiles is a chain that every K block repeats (barrier, the burst of LDS reads behind it,
// MFMAs, barrier): 333 x 4096 x 7168 block-FP8 takes 24.7 us, 19.5 without any copy behind the first stages, 23.4 without the
// MFMAs, 23.3 without the LDS reads.  Here nothing is shared until the end:
//   * each of the block's four waves computes the whole tile on every fourth K block, from a ring of its own in LDS that it
//     fills itself: no barrier in the loop, a wave waits for its own copies only, and every operand byte is read from LDS once
//     (the ring's eight waves read a 64 x 128 tile's 24 KiB K block as 64 KiB);
//   * the ring's slots are units of 32 rows (4 KiB), refilled as soon as the MFMAs that use their fragments have been issued:
//     behind a step's refills 80-128 KiB per CU are under way, across a wait 32-96 KiB, two of a wave's units at least;
//   * one wave per SIMD has all of its registers: 48-192 accumulators, the K block's activations, two units of weights.
// The partial sums meet in LDS, added in the order of the waves.
// Bound now: what a CU takes in past the L2, 60-70 GB/s with HBM latency (a build that only copies is as fast; one whose copies
// hit the L2 takes 0.22 instead of 0.33 us per K block of 64 x 128), and the fixed 3.5-6 us of launch, ring fill and reduction.
// Measured (graph-timed, weights from HBM, the kernel that took it before -> here): block-FP8 630 x 1280 x 4608 15.3 -> 10.9 us,
// 512 x 2112 x 7168 23.3 -> 21.0, 333 x 4096 x 7168 25.9 -> 24.5, per-token FP8 277 x 2112 x 6400 16.2 -> 12.1, INT8
// 506 x 1920 x 8576 23.7 -> 16.8.  Tried and not kept: another order of K blocks for each row tile of a weight tile
// (512 x 2112 x 7168 23.4 -> 21.0, but 200 x 8192 x 8192 29.2 -> 41.4: the weights leave the L2 before they are read again), a fifth
// wave that fetches weight rows into the L2 (up to 8 % on 96 x 64 tiles, nothing on the others).
#pragma once
#include "gemm_device.h"

namespace sglq {

// The tile shapes that are built: X(index, MI, NI).  16 MI rows, 16 NI columns.
#define SGLQ_KWAVE_CONFIGS(X) \
  X(0, 2, 4)                  \
  X(1, 3, 4)                  \
  X(2, 4, 4)                  \
  X(3, 5, 4)                  \
  X(4, 6, 4)                  \
  X(5, 7, 4)                  \
  X(6, 2, 8)                  \
  X(7, 3, 8)                  \
  X(8, 4, 8)                  \
  X(9, 8, 4)                  \
  X(10, 6, 8)
constexpr int KWAVE_CONFIGS = 11;
#define SGLQ_KWAVE_BM(i, mi, ni) 16 * mi,
#define SGLQ_KWAVE_BN(i, mi, ni) 16 * ni,
constexpr int KWAVE_BM[] = {SGLQ_KWAVE_CONFIGS(SGLQ_KWAVE_BM)};
constexpr int KWAVE_BN[] = {SGLQ_KWAVE_CONFIGS(SGLQ_KWAVE_BN)};
// The kinds that fold every MFMA's result into the accumulators keep these in the 256 registers that vector instructions
// reach and are built where these suffice without scratch; the others accumulate in the other 256.
constexpr bool kwave_built(int kind, int config) { return (config != 5 && config < 9) || !(kind == KIND_FP8_BLOCK || kind == KIND_I8_BLOCK); }

void launch_kwave_fp8_block(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_kwave_fp8_rowcol(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_kwave_i8_rowcol(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_kwave_i8_block(GemmArgs& p, int config, int out_dtype, hipStream_t st);

}  // namespace sglq
