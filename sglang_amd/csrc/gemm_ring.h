// gemm_ring_kernel: the GEMM for 17 to a few thousand rows, where the 256-row kernels would leave most of the chip
// idle and the weight-streaming kernels re-read their operands too often.
//
// What bounds these shapes is not arithmetic but what a compute unit takes in: its global -> LDS copies deliver about
// 64-70 GB/s while the lines come from HBM, 90-100 from the last-level cache and at most 150 (64 bytes a clock) from
// the XCD's L2, whatever their number (measured with copies alone: deeper rings, more copying waves and cache hints
// change nothing; what is in flight per CU is capped).  So the tile is chosen for the least operand bytes per CU, with
// one block on every CU and K not split, and the kernel is built so that the copies never stop:
//   * four producer waves issue nothing but copies (a copy's issue blocks while the address unit is busy; in a wave
//     that also multiplies, that time is lost to the matrix pipe: a 64 x 64 tile's K block took 0.31 us in
//     gemm_stream_kernel, where every wave copies for itself);
//   * eight consumer waves read operands from a ring of NST stages and multiply.  One barrier per stage: in front of
//     it a producer waits for the next stage's copies (its oldest ones; vector-memory operations retire in order) and
//     a consumer for its last LDS reads of the current stage; behind it the stage is refilled.  The consumers' first
//     fragments of a stage are read behind that barrier, under the last MFMAs of the stage before.
// Waves: WM x WN over the tile, each with MI x NI fragments of 16 x 16, times KG groups that take alternate K blocks
// (a stage holds KG K blocks; their partial sums meet in LDS at the end, in group order).  The operand with fewer
// fragments is held in registers for a K block, the other one streams through two fragments: 69-134 registers, three
// waves per SIMD.
// Measured (weights in turn from more than the last-level cache; before -> after): block-FP8 64 x 57344 x 8192
// 102 -> 92 us, 333 x 4096 x 7168 26.7 (split K, two launches) -> 24, 466 x 2816 x 3456 17 -> 11.3, block-INT8
// 1000 x 5120 x 5120 46 -> 35.
#pragma once
#include "gemm_device.h"

namespace sglq {

// The tile shapes that are built: X(index, WM, WN, KG, MI, NI, NST).  BM = 16 WM MI rows, BN = 16 WN NI columns.
#define SGLQ_RING_CONFIGS(X) \
  X(0, 4, 1, 2, 1, 1, 6)     \
  X(1, 4, 1, 2, 1, 2, 6)     \
  X(2, 4, 1, 2, 1, 3, 5)     \
  X(3, 2, 2, 2, 2, 2, 4)     \
  X(4, 4, 2, 1, 1, 3, 6)     \
  X(5, 2, 4, 1, 2, 2, 6)     \
  X(6, 4, 2, 1, 1, 6, 4)     \
  X(7, 4, 2, 1, 1, 7, 4)     \
  X(8, 2, 4, 1, 4, 1, 5)     \
  X(9, 4, 2, 1, 2, 3, 5)     \
  X(10, 2, 4, 1, 4, 2, 4)    \
  X(11, 4, 2, 1, 2, 5, 4)    \
  X(12, 4, 2, 1, 2, 6, 3)    \
  X(13, 2, 4, 1, 4, 4, 3)    \
  X(14, 2, 1, 4, 1, 2, 4)    \
  X(15, 2, 2, 2, 1, 2, 5)
constexpr int RING_CONFIGS = 16;
#define SGLQ_RING_BM(i, wm, wn, kg, mi, ni, nst) 16 * wm * mi,
#define SGLQ_RING_BN(i, wm, wn, kg, mi, ni, nst) 16 * wn * ni,
#define SGLQ_RING_KG(i, wm, wn, kg, mi, ni, nst) kg,
constexpr int RING_BM[] = {SGLQ_RING_CONFIGS(SGLQ_RING_BM)};
constexpr int RING_BN[] = {SGLQ_RING_CONFIGS(SGLQ_RING_BN)};
constexpr int RING_KG[] = {SGLQ_RING_CONFIGS(SGLQ_RING_KG)};

// ... and whether a grouped (expert) GEMM is built on it
constexpr bool RING_GROUPED[] = {false, false, false, false, false, true, false, false, false, false, false, false, false, false, false, false};

// Launches configuration `config` for the problem (tiles_m / tiles_n are set here); one function per kind, each in a
// translation unit of its own.
void launch_ring_fp8_block(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_ring_fp8_block_grouped(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_ring_fp8_block_pow2(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_ring_fp8_rowcol(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_ring_i8_rowcol(GemmArgs& p, int config, int out_dtype, hipStream_t st);
void launch_ring_i8_block(GemmArgs& p, int config, int out_dtype, hipStream_t st);

}  // namespace sglq
