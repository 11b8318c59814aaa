// gemm_kwave_kernel: the GEMM for 17 to some two thousand rows with small tiles, K split over the waves of a block.
//
// What bounds gemm_ring_kernel on such tiles is a chain that every K block repeats (barrier, the burst of LDS reads behind it,
// MFMAs, barrier): 333 x 4096 x 7168 block-FP8 took 24.7 us, 19.5 without any copy behind the first stages, 23.4 without the
// MFMAs, 23.3 without the LDS reads, all in one run.  Here nothing is shared until the end:
//   * each of the block's four waves computes the whole tile on every fourth K block, from a ring of its own in LDS that it
//     fills itself: no barrier in the loop, a wave waits for its own copies only, and every operand byte is read from LDS once
//     (the ring's eight waves read a 64 x 128 tile's 24 KiB K block as 64 KiB);
//   * the ring's slots are units of 32 rows (4 KiB), refilled as soon as the MFMAs that use their fragments have been issued:
//     behind a step's refills 80-128 KiB per CU are under way, across a wait 32-96 KiB, two of a wave's units at least;
//   * one wave per SIMD has all of its registers: 48-192 accumulators, the K block's activations, two units of weights.
// The partial sums meet in LDS, added in the order of the waves.
// Bound now: operand intake, 55-65 GB/s per CU with the weights from HBM whatever the tile and however few CUs run (a build that only
// copies is as fast; one whose copies hit the L2 takes 0.22 instead of 0.33 us per K block of 64 x 128), and the fixed 3.5-6 us of
// launch, ring fill and reduction.  It is not the copy path's limit: a bare copy loop takes in 118-124 GB/s from windows that four
// blocks share; what holds the copies here to half of that is not known.
// Measured (graph-timed, one run; the kernel that took it before -> here with the weights from HBM, and with the weight in the
// last-level cache): block-FP8 333 x 4096 x 7168 25.0 -> 21.1 and 22.4 -> 18.9 us, 512 x 2112 x 7168 23.4 -> 18.7 and 22.1 -> 16.2,
// 630 x 1280 x 4608 15.0 -> 12.5 and 15.3 -> 10.8, per-token FP8 277 x 2112 x 6400 16.6 -> 14.2 and 16.2 -> 9.7, INT8
// 506 x 1920 x 8576 23.0 -> 19.7 and 22.1 -> 16.8.  Tried and not kept: another order of K blocks for each row tile of a weight tile
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
