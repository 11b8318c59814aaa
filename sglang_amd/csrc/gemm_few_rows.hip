// gemm_few_rows_kernel: GEMM 1 of an expert layer of few rows an expert (decode) on 32- or 64-row tiles, with the activation and its quantization behind it.
//
// Bound by the weights' bytes from HBM.  A tile is 32 or 64 rows x 128 gates and their 128 partners, so that it holds whole groups of the activation; half as many tiles as
// gemm_kernel<32 x 128> and the ring's 64 x 128 have.  Two blocks of two stages a CU, as gemm_kernel has four, drain at every K block and lose on few tiles what the launch saves
// (16 experts, 5120 x 1536, 192 tiles: 86.6 -> 97.4 us a layer); so one block a CU keeps four stages of 37 KiB, three of them in flight (64 rows: three of 41, two), and walks its tiles without a
// break: the copies run on into the next tile while one is finished.  Eight waves copy, five or six operations a stage each, and multiply, 16 gates and 16 partners each.
// Layers without and with it, us (tokens x experts x top-k, hidden x intermediate), on 32 rows: 16 x 32 x 8, 7168 x 2048 242.7 -> 231.2; 32 x 64 x 8, 4096 x 1024 147.3 -> 138.4;
// 16 x 16 x 4, 5120 x 1536 86.9 -> 81.2; 42 x 64 x 6, 2048 x 1408 112.3 -> 106.4; 128 x 128 x 8, 2048 x 768 121.3 -> 114.3; on 64 rows: 480 x 60 x 4, 2048 x 1408 146.8 -> 129.3; 100 x 16 x 4,
// 5120 x 1536 109.6 -> 97.8; 512 x 128 x 8, 2048 x 768 173.1 -> 156.5.  GEMM 2 on the same loop (256 columns and four stages, or 128 and seven) is 1 to 3 % slower than on gemm_kernel
// and stays there.
#include "gemm_device.h"
#include "gemm_few_rows.h"
#include "quant_device.h"
#include "silu_device.h"

namespace sglq {

constexpr int FEW_WAVES = 8;

template <int OUT_DT, int BM>
__global__ __launch_bounds__(FEW_WAVES * 64, 2) void gemm_few_rows_kernel(const GemmArgs p) {
  static_assert(BM == 32 || BM == 64, "four or eight copies of activations a stage");
  constexpr int NW = FEW_WAVES, BN = 256, NST = BM == 32 ? 4 : 3, MI = BM / 16, NI = 2, BCOPIES = BN / 8 / NW;
  constexpr int CPS = BCOPIES + BM / 32;  // copies of a wave and stage: its part of the weights, and one of the rest (64 rows: one of the activations and one of the rest)
  constexpr int W_SCALES = BM == 32 ? 4 : 0;  // the wave that copies the activations' scales; the next one copies the weights'
  constexpr int STAGE_BYTES = (BM + BN) * 128 + 512, SCALES = (BM + BN) * 128;
  constexpr int DUMP = NST * STAGE_BYTES, CODES = DUMP + 256, MAXIMA = CODES + BM * 128;
  static_assert((NST - 2) * CPS < 64, "vmcnt holds six bits");
  constexpr int LDS = MAXIMA + BM * NW * 2;
  static_assert(LDS <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) char smem[LDS];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4, l8 = lane >> 3;
  const int* const plan = static_cast<const int*>(p.ws);
  const int listed = plan[0], tiles_m = listed < p.tiles_m ? listed : p.tiles_m;
  const int total = tiles_m * p.tiles_n, nkb = p.K >> 7, half = p.N >> 1;
  const uint32_t base = lds_addr(smem);
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ l8 ^ (wave & 1)) & 7) * 16u;  // (copies of a wave are eight groups of rows apart)
  const int nblocks = (p.N + 127) >> 7;
  const uint32_t sa_bytes = (uint32_t)(((int64_t)(p.M - 1) * p.sa_stride_m + (int64_t)(nkb - 1) * p.sa_stride_k + 1) * 4);
  const uint32_t sb_bytes = (uint32_t)(((int64_t)(nblocks - 1) * p.sb_stride_n + (int64_t)(nkb - 1) * p.sb_stride_k + 1) * 4);
  const v4u ra = make_rsrc_sgpr(p.a, p.a_bytes), rsa = make_rsrc_sgpr(p.sa, sa_bytes);
  const int sw = (r16 & 7) ^ (r16 >> 3);
  const int lane_off0 = r16 * 128 + (((2 * g) ^ sw) * 16), lane_off1 = lane_off0 ^ 16;
  const int mine = total > (int)blockIdx.x ? (total - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;

  for (int from = 0; from < mine; from += 64) {  // (64 tiles of the block, one to a lane)
    const int here = mine - from < 64 ? mine - from : 64;
    int t_m0 = 0, t_end = 0, t_expert = 0, t_n = 0;
    if (lane < here) {
      int tm;
      tile_of_block((int)blockIdx.x + (from + lane) * (int)gridDim.x, tiles_m, p.tiles_n, tm, t_n);
      const int* entry = plan + PLAN_HEADER + PLAN_ENTRY * tm;
      t_expert = entry[0];
      t_m0 = entry[1];
      t_end = entry[2];
    }
    __builtin_amdgcn_s_waitcnt(0);

    // ---- copies: the stage of a step holds its K block's activations, weights and scales
    int c_tile = -1, c_left = 0, c_kb = 0;
    v4u rb = ra, rsb = ra;
    uint32_t off_b[BCOPIES], off_a = OOB, off_s = OOB;
#pragma unroll
    for (int j = 0; j < BCOPIES; ++j) off_b[j] = OOB;
    auto next_tile = [&]() {
      ++c_tile;
      c_left = nkb;
      if (c_tile >= here) {
        c_left = 1 << 30;
        off_a = off_s = OOB;
#pragma unroll
        for (int j = 0; j < BCOPIES; ++j) off_b[j] = OOB;
        return;
      }
      const int m0 = __builtin_amdgcn_readlane(t_m0, c_tile), end = __builtin_amdgcn_readlane(t_end, c_tile);
      const int expert = __builtin_amdgcn_readlane(t_expert, c_tile), tn = __builtin_amdgcn_readlane(t_n, c_tile);
      rb = make_rsrc_sgpr(p.b + (int64_t)expert * p.b_expert_stride, p.b_bytes);
      rsb = make_rsrc_sgpr(p.sb + (int64_t)expert * p.sb_expert_stride, sb_bytes);
      c_kb = __builtin_amdgcn_readfirstlane(first_k_step(p, grouped_weight_tile(p, expert, tn), nkb));
#pragma unroll
      for (int j = 0; j < BCOPIES; ++j) {
        const int c = wave + NW * j;  // rows 8 c .. of the stage's weights
        const int col = tn * (BN / 2) + (c >> 2) * 16 + (c & 1) * 8 + l8 + (c & 2 ? half : 0);  // 16 gates of a wave, 16 partners
        off_b[j] = (uint32_t)col * p.ldb + chunk;
      }
      const int row = m0 + wave * 8 + l8;
      off_a = (BM == 64 || wave < 4) && row < end ? (uint32_t)row * p.lda + chunk : OOB;
      off_s = OOB;
      if (wave == W_SCALES) {
        if (lane < BM && m0 + lane < end) off_s = (uint32_t)((m0 + lane) * p.sa_stride_m * 4);
      } else if (wave == W_SCALES + 1) {
        if (lane < 2) off_s = (uint32_t)((tn + (lane ? half >> 7 : 0)) * p.sb_stride_n * 4);
      }
    };
    auto issue = [&](int slot) {
      if (c_left == 0) next_tile();
      const uint32_t st = base + (uint32_t)slot * STAGE_BYTES, kb = (uint32_t)c_kb;
      const bool live = c_tile < here;
#pragma unroll
      for (int j = 0; j < BCOPIES; ++j) lds_copy16(rb, st + BM * 128 + (uint32_t)(wave + NW * j) * 1024u, off_b[j], live ? kb * 128u : 0u);
      if (BM == 64 || wave < 4) lds_copy16(ra, st + (uint32_t)wave * 1024u, off_a, live ? kb * 128u : 0u);
      if (BM == 64 || wave >= 4) {
        if (wave == W_SCALES) lds_copy4(rsa, st + SCALES, off_s, live ? kb * (uint32_t)(p.sa_stride_k * 4) : 0u);
        else if (wave == W_SCALES + 1) lds_copy4(rsb, st + SCALES + 256, off_s, live ? kb * (uint32_t)(p.sb_stride_k * 4) : 0u);
        else lds_copy4(rsa, base + DUMP, OOB, 0u);
      }
      --c_left;
      c_kb = c_kb + 1 == nkb ? 0 : c_kb + 1;
    };
    int fill = 0, slot = 0;
#pragma unroll
    for (int s = 0; s < NST - 1; ++s) issue(fill++);

    for (int tile = 0; tile < here; ++tile) {
      v4f acc[MI][NI];
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = v4f{0, 0, 0, 0};
      for (int step = 0; step < nkb; ++step) {
        __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0_only());  // the stage before is read
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * CPS) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(fill);
        fill = fill + 1 == NST ? 0 : fill + 1;
        const char* st = smem + slot * STAGE_BYTES;
        slot = slot + 1 == NST ? 0 : slot + 1;
        float sfa[MI];
        v8i af[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const char* q = st + i * 16 * 128;
          const v4i lo = *reinterpret_cast<const v4i*>(q + lane_off0), hi = *reinterpret_cast<const v4i*>(q + lane_off1);
          af[i] = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          sfa[i] = *reinterpret_cast<const float*>(st + SCALES + (i * 16 + r16) * 4);
        }
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const char* q = st + (BM + (wave * NI + j) * 16) * 128;
          const v4i lo = *reinterpret_cast<const v4i*>(q + lane_off0), hi = *reinterpret_cast<const v4i*>(q + lane_off1);
          const v8i bf = v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          const float sfb = *reinterpret_cast<const float*>(st + SCALES + 256 + j * 4);
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const v4f part = block_mfma<KIND_FP8_BLOCK>(bf, af[i]);
            const float sc = sfa[i] * sfb;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(part[e], sc, acc[i][j][e]);
          }
        }
      }
      const int m0 = __builtin_amdgcn_readlane(t_m0, tile), end = __builtin_amdgcn_readlane(t_end, tile), tn = __builtin_amdgcn_readlane(t_n, tile);
      uint16_t* const maxima = reinterpret_cast<uint16_t*>(smem + MAXIMA);  // [BM rows][8 waves]
      uint32_t h[MI][2];
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const uint32_t m = silu_of_rows<OUT_DT, 1>(acc[i], h[i]);
        if (g == 0) maxima[(i * 16 + r16) * NW + wave] = (uint16_t)m;
      }
      __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0_only());
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const int row = i * 16 + r16;
        const v4u eight = *reinterpret_cast<const v4u*>(maxima + row * NW);
        const float y_s = silu_scale<OUT_DT>(eight, p.quant_eps), inv = 1.0f / y_s;
        *reinterpret_cast<uint32_t*>(smem + CODES + row * 128 + wave * 16 + g * 4) = silu_codes<OUT_DT>(h[i][0], h[i][1], y_s, inv);
        if (wave == i && g == 0 && m0 + row < end) p.out_scales[(int64_t)tn * p.M + m0 + row] = y_s;
      }
      __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0_only());
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const int row = threadIdx.x >> 3, at = (threadIdx.x & 7) * 16;
      if (row < BM && m0 + row < end)
        *reinterpret_cast<v4u*>(reinterpret_cast<char*>(p.out) + (int64_t)(m0 + row) * half + tn * 128 + at) = *reinterpret_cast<const v4u*>(smem + CODES + row * 128 + at);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no copy outlives the tiles it was for)
    __builtin_amdgcn_s_barrier();
  }
}

void launch_few_rows(GemmArgs& p, int max_tiles, int rows, int out_dtype, hipStream_t st) {
  p.tiles_m = max_tiles;
  p.tiles_n = p.N / 256;
  p.splits = 1;
  const int64_t tiles = (int64_t)max_tiles * p.tiles_n;
  const dim3 grid((uint32_t)(tiles < p.cus ? tiles : p.cus)), block(FEW_WAVES * 64);
  if (rows == 32 && out_dtype == SGLQ_BF16) gemm_few_rows_kernel<SGLQ_BF16, 32><<<grid, block, 0, st>>>(p);
  else if (rows == 32) gemm_few_rows_kernel<SGLQ_FP16, 32><<<grid, block, 0, st>>>(p);
  else if (out_dtype == SGLQ_BF16) gemm_few_rows_kernel<SGLQ_BF16, 64><<<grid, block, 0, st>>>(p);
  else gemm_few_rows_kernel<SGLQ_FP16, 64><<<grid, block, 0, st>>>(p);
}

}  // namespace sglq
