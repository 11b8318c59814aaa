// The data movement around the grouped (MoE) block-scaled FP8 GEMM on gfx950: routing
// tables from the top-k expert ids, row gathers into expert-major order, SiLU-and-multiply
// between the two GEMMs, and the weighted combine back to token order.  All HBM-bound.
#include <type_traits>

#include "gemm_device.h"
#include "quant_device.h"
#include "sglq_common.h"

namespace sglq {

static int check_moe_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return SGLQ_ELAUNCH;
  }
  return SGLQ_OK;
}

// ---------------------------------------------------------------------------
// prepare_moe_input (sgl-kernel/csrc/moe/prepare_moe_input.cu:13-139): from topk_ids
// [topk_length] (token-major: slot i belongs to token i / topk) build
//   problem_sizes1[e] = (count_e, 2 n, k), problem_sizes2[e] = (count_e, k, n)       (:31-38)
//   expert_offsets[0 .. E] = running sum of the counts                                (:41-54)
//   blockscale_offsets[0 .. E] (optional) = running sum of the counts rounded up to 128 (:56-76)
//   input_permutation[p] = token of the slot that lands in expert-major position p     (:93)
//   output_permutation[i] = expert-major position of slot i                            (:94)
// The reference hands out positions inside an expert with atomicAdd, in whatever order the
// threads arrive; here slots keep their order (position = number of earlier slots of the same
// expert), so the tables are the same on every run.  Ids outside [0, E) belong to nobody: their
// output_permutation entries are left as they are, as in the reference.
// The counts of every expert must be known before any offset, hence three launches: count
// (one block per expert), offsets (one block scanning E values), place.  A thread looks at
// four consecutive slots at a time, a block of 1024 threads at 4096.
// ---------------------------------------------------------------------------
constexpr int MOE_THREADS = 1024, MOE_SWEEP = 4 * MOE_THREADS;

// Slots i .. i + 3; slots past the end read as -1, which is nobody's id.
SGLQ_DEV v4i load_ids4(const int* __restrict__ ids, int64_t i, int64_t n, bool aligned) {
  if (aligned && i + 3 < n) return *reinterpret_cast<const v4i*>(ids + i);
  v4i v = {-1, -1, -1, -1};
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (i + q < n) v[q] = ids[i + q];
  return v;
}

// Number of slots in [0, end) that name expert e; every thread of the block gets the sum.
SGLQ_DEV int block_count_ids(const int* __restrict__ ids, int64_t end, int e, bool aligned, int* red) {
  int c = 0;
#pragma unroll 4
  for (int64_t i = 4 * (int64_t)threadIdx.x; i < end; i += MOE_SWEEP) {
    const v4i v = load_ids4(ids, i, end, aligned);
    c += (v[0] == e) + (v[1] == e) + (v[2] == e) + (v[3] == e);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) c += __shfl_xor(c, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  c = 0;
#pragma unroll
  for (int w = 0; w < MOE_THREADS / 64; ++w) c += red[w];
  __syncthreads();
  return c;
}

__global__ __launch_bounds__(MOE_THREADS) void moe_count_kernel(const int* __restrict__ topk_ids, int* __restrict__ ps1,
                                                                int* __restrict__ ps2, int64_t topk_length, int n, int k,
                                                                int aligned) {
  __shared__ int red[MOE_THREADS / 64];
  const int e = blockIdx.x;
  const int c = block_count_ids(topk_ids, topk_length, e, aligned != 0, red);
  if (threadIdx.x == 0) {
    ps1[3 * e] = c;
    ps1[3 * e + 1] = 2 * n;
    ps1[3 * e + 2] = k;
    ps2[3 * e] = c;
    ps2[3 * e + 1] = k;
    ps2[3 * e + 2] = n;
  }
}

__global__ __launch_bounds__(256) void moe_offsets_kernel(const int* __restrict__ ps1, int* __restrict__ expert_offsets,
                                                          int* __restrict__ blockscale_offsets, int num_experts) {
  __shared__ int scan[256], scan_r[256];
  __shared__ int base, base_r;
  const int tid = threadIdx.x;
  if (tid == 0) {
    base = 0;
    base_r = 0;
    expert_offsets[0] = 0;
    if (blockscale_offsets) blockscale_offsets[0] = 0;
  }
  __syncthreads();
  for (int e0 = 0; e0 < num_experts; e0 += 256) {
    const int e = e0 + tid;
    const int c = e < num_experts ? ps1[3 * e] : 0;
    const int r = (c + 127) / 128 * 128;
    scan[tid] = c;
    scan_r[tid] = r;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {
      const int v = tid >= d ? scan[tid - d] : 0, vr = tid >= d ? scan_r[tid - d] : 0;
      __syncthreads();
      scan[tid] += v;
      scan_r[tid] += vr;
      __syncthreads();
    }
    if (e < num_experts) {
      expert_offsets[e + 1] = base + scan[tid];
      if (blockscale_offsets) blockscale_offsets[e + 1] = base_r + scan_r[tid];
    }
    __syncthreads();
    if (tid == 255) {
      base += scan[255];
      base_r += scan_r[255];
    }
    __syncthreads();
  }
}

// Block (e, part) places expert e's slots of the part-th range of `span` slots (a multiple of
// 4096); it first counts the expert's slots in the ranges before its own, which is where its
// positions start.  Inside a sweep a slot's position follows from the matches before it:
// those of earlier waves, of earlier lanes of its wave (one ballot per slot of the four), and
// of the thread's own earlier slots.
__global__ __launch_bounds__(MOE_THREADS) void moe_place_kernel(const int* __restrict__ topk_ids,
                                                                const int* __restrict__ expert_offsets,
                                                                int* __restrict__ input_permutation,
                                                                int* __restrict__ output_permutation, int64_t topk_length,
                                                                int topk, int64_t span, int aligned) {
  __shared__ int red[MOE_THREADS / 64];
  __shared__ int wave_count[2][MOE_THREADS / 64];
  const int e = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t begin = (int64_t)blockIdx.y * span;
  if (begin >= topk_length) return;
  const int64_t end = begin + span < topk_length ? begin + span : topk_length;
  int next = expert_offsets[e] + block_count_ids(topk_ids, begin, e, aligned != 0, red);
  const uint64_t below = (1ull << lane) - 1ull;
  int buf = 0;
  v4i v = load_ids4(topk_ids, begin + 4 * (int64_t)threadIdx.x, end, aligned != 0);
  for (int64_t i0 = begin; i0 < end; i0 += MOE_SWEEP, buf ^= 1) {
    const int64_t i = i0 + 4 * (int64_t)threadIdx.x;
    const v4i cur = v;
    if (i0 + MOE_SWEEP < end) v = load_ids4(topk_ids, i + MOE_SWEEP, end, aligned != 0);  // the next sweep's, ahead of the barrier
    int before = 0, in_wave = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint64_t ballot = __ballot(cur[q] == e);
      before += __popcll(ballot & below);
      in_wave += __popcll(ballot);
    }
    if (lane == 0) wave_count[buf][wave] = in_wave;
    __syncthreads();  // (the buffer written two sweeps ago was last read before the previous sweep's barrier)
    int earlier_waves = 0, total = 0;
#pragma unroll
    for (int w = 0; w < MOE_THREADS / 64; ++w) {
      const int c = wave_count[buf][w];
      earlier_waves += w < wave ? c : 0;
      total += c;
    }
    int pos = next + earlier_waves + before;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (cur[q] == e) {
        input_permutation[pos] = (int)((i + q) / topk);
        output_permutation[i + q] = pos;
        ++pos;
      }
    }
    next += total;
  }
}

// ---------------------------------------------------------------------------
// The same tables, the -1 default of output_permutation and the grouped GEMMs' tile plan in one launch,
// for up to 32768 slots and 512 experts.  A decode step's layer is a chain of short dependent launches,
// each of 2-5 us whatever it does (16 tokens, 32 experts: the fill of c_map, the three launches above and
// two plan launches were 28 of the layer's 273 us).
// A block places the slots of one segment.  Sixteen waves take consecutive ranges of it and keep their ids in registers; counts per
// (wave, expert) through LDS atomics (sums: the order does not matter), a running sum over waves and experts, then every
// wave walks its slots again in order: lanes that name the same expert find each other with one ballot per
// id bit, so positions follow slot order as above.  That walk is a chain of LDS round trips, 64 slots of a wave at a time, and what a long
// prompt's tables spent their time on; so above 2048 slots there are several segments, and each block counts all slots
// for itself, which needs no exchange between blocks: a slot adds 1 to its expert's word, and 65536 more where it lies in front
// of the block's segment.  One block -> segments of 1024 slots (us): 5600 slots of 64 experts 9.7 -> 7.3, 20000 of 32 17.5 -> 9.3, 32768 of 32
// 24.7 -> 11.3 (of 2048 slots 11.8, of 4096 12.9); 128 slots, where no step that there are no slots for is walked any more, 6.5 -> 5.7.
// ---------------------------------------------------------------------------
constexpr int TABLE_THREADS = 1024, TABLE_WAVES = TABLE_THREADS / 64, TABLE_STEPS = 32;
constexpr int TABLE_MAX_SLOTS = TABLE_THREADS * TABLE_STEPS, TABLE_MAX_EXPERTS = 512;
// (several segments double the LDS: 32 KiB at 256 experts, from there on one)
constexpr int TABLE_ONE_SEGMENT = 2048, TABLE_SEGMENT = TABLE_THREADS, TABLE_SEGMENTS_EXPERTS = 256;

// The walks of the layer's two GEMMs on 256-row tiles (gemm_device.h), written by blocks of their own, which count the slots as the others do and place
// none: a band is an expert's row tiles, up to WALK_BAND of them (of more than that bands of like size), column by column, so that the blocks of an XCD share the
// weights that they read at the same time and every weight is read by one band only.
struct LayerWalks {
  int* walk[2];
  FastDiv columns[2];  // column tiles
  int first_block;     // blocks from here on write them (none: the grid ends there)
};
constexpr int WALK_BAND = 8, WALK_ROWS = 256;

// The activations of a layer of few slots, quantized beside its tables by blocks of their own; codes and scales are group_quant_scatter_kernel's (quant.hip; CM, ONCE).
// Both launches are latency (tables 5.4 us, quantization 4.1-5.0 behind each other, whatever they hold), and the blocks depend on the ids alone.
struct LayerQuant {
  const char* x;
  char* q;
  float* s;
  FastDiv walk;  // blocks to a band of tokens
  uint32_t num_tokens, groups_per_row;
  int first_block;  // blocks from here on (none: the grid ends there)
  float eps, qmax, rqmax;
};
constexpr int QUANT_STEPS = 32, QUANT_MAX_SLOTS = 64 * QUANT_STEPS, QUANT_MAX_TOPK = 64;
constexpr int QUANT_TOKENS = 2, QUANT_WAVES = TABLE_WAVES / QUANT_TOKENS;  // tokens to a block, waves to a token

// A wave takes eight groups of 128 of one token.  Where the token's slots go its waves find for themselves, since the tables are being written: slots ordered by
// (expert, slot) lie where their rank says, so a lane keeps such keys of every 64th slot and a ballot a step counts those in front.  Eight waves share a token's
// slots (of a layer of 512 and of 1024 slots of 8 x 2, 6144 x 2048, us without / so: 106.8 / 102.7, 123.9 / 121.7; every wave for itself 16 tokens a block 109.4 / 105.7 and
// 128.3 / 124.1, but 128 tokens x 128 x 8, 2048 x 768 125.9 -> 128.0 instead of 120.5; a band of 16 tokens placed by the tables' own code 0 to 2 us of the 4 won).
template <int DT, bool ONCE>
SGLQ_DEV void quantize_beside_tables(const int* __restrict__ topk_ids, int topk, int topk_length, int num_experts, const LayerQuant& quant,
                                     int (&slot_row)[QUANT_TOKENS][QUANT_MAX_TOPK]) {
  constexpr uint32_t NOBODY = ~0u;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t t = wave / QUANT_WAVES, of_token = wave % QUANT_WAVES, sub = lane & 7;
  const uint32_t b = blockIdx.x - (uint32_t)quant.first_block, band = quant.walk.div(b);
  const uint32_t token = band * QUANT_TOKENS + t, group = ((b - band * quant.walk.d) * QUANT_WAVES + of_token) * 8 + (lane >> 3);
  const bool there = token < quant.num_tokens, live = there && group < quant.groups_per_row;
  const int64_t hidden = (int64_t)quant.groups_per_row * 128, at = (int64_t)group * 128 + sub * 8;
  Chunk8<DT> ch[2];
  if (live) {
#pragma unroll
    for (int c = 0; c < 2; ++c) ch[c].load(quant.x + (token * hidden + at + c * 64) * elem_bytes<DT>());
  }
  const int steps = (topk_length + 63) >> 6;
  auto key_of = [&](int i, bool any) {
    const uint32_t e = any ? (uint32_t)topk_ids[i] : NOBODY;
    return e < (uint32_t)num_experts ? e * QUANT_MAX_SLOTS + (uint32_t)i : NOBODY;
  };
  const uint32_t own = key_of((int)token * topk + lane, there && lane < topk);
  uint32_t keys[QUANT_STEPS];
#pragma unroll
  for (int s = 0; s < QUANT_STEPS; ++s) keys[s] = key_of(s * 64 + lane, s * 64 + lane < topk_length);
  for (int j = (int)of_token; j < topk; j += QUANT_WAVES) {
    const uint32_t key = (uint32_t)__builtin_amdgcn_readlane((int)own, j);
    int row = 0;
#pragma unroll
    for (int s = 0; s < QUANT_STEPS; ++s) {
      if (s >= steps) break;
      row += __popcll(__ballot(keys[s] < key));
    }
    slot_row[t][j] = key == NOBODY ? -1 : row;
  }
  v2u o[2];
  float y_s = 0.f;
  if (live) {
    const uint32_t mb = group_umax<8>(umax(ch[0].amax_bits(), ch[1].amax_bits()));
    const float amax = u2f(umax(mb, f2u(quant.eps)));
    y_s = div_by(amax, quant.qmax, quant.rqmax);
    const float r = 1.0f / y_s;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = quantize_elem<false>(ch[c].get(i), y_s, r, -quant.qmax, quant.qmax);
      o[c] = Fp8Pack::pack(v);
    }
  }
  __syncthreads();
  if (!live) return;
  if constexpr (ONCE) {
#pragma unroll
    for (int c = 0; c < 2; ++c) *reinterpret_cast<v2u*>(quant.q + token * hidden + at + c * 64) = o[c];
  }
  for (int j = ONCE ? (int)sub : 0; j < topk; j += ONCE ? 8 : 1) {
    const int row = slot_row[t][j];
    if (row < 0) continue;
    if constexpr (!ONCE) {
#pragma unroll
      for (int c = 0; c < 2; ++c) *reinterpret_cast<v2u*>(quant.q + row * hidden + at + c * 64) = o[c];
    }
    if (ONCE || sub == 0) quant.s[(int64_t)group * topk_length + row] = y_s;
  }
}

// QUANT_DT: the activations' type, -1: tables only
template <int QUANT_DT, bool ONCE>
__global__ __launch_bounds__(TABLE_THREADS) void moe_tables_kernel(const int* __restrict__ topk_ids, int* __restrict__ expert_offsets,
                                                                   int* __restrict__ ps1, int* __restrict__ ps2,
                                                                   int* __restrict__ output_permutation, int* __restrict__ input_permutation,
                                                                   FastDiv topk, int topk_length, int num_experts, int id_bits, int n, int k, int* __restrict__ plan,
                                                                   int plan_rows, int plan_max_tiles, int segment, const LayerWalks walks,
                                                                   const LayerQuant quant) {
  if constexpr (QUANT_DT >= 0) {
    if ((int)blockIdx.x >= quant.first_block) {
      __shared__ int slot_row[QUANT_TOKENS][QUANT_MAX_TOPK];
      quantize_beside_tables<QUANT_DT, ONCE>(topk_ids, (int)topk.d, topk_length, num_experts, quant, slot_row);
      return;
    }
  }
  // [TABLE_WAVES][num_experts]: first the segment's counts, then the next position of each; of several segments, all slots' behind them
  extern __shared__ int counts[];
  __shared__ int wave_rows[TABLE_WAVES], wave_tiles[TABLE_WAVES];
  __shared__ int expert_rows[TABLE_MAX_EXPERTS], expert_end[TABLE_MAX_EXPERTS], expert_tiles[TABLE_MAX_EXPERTS];  // (walks only)
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int begin_slot = (int)blockIdx.x * segment, end_slot = begin_slot + segment < topk_length ? begin_slot + segment : topk_length;
  const bool alone = quant.first_block == 1;
  const int steps = segment / TABLE_THREADS;  // 64 slots each, per wave
  const int first = begin_slot + wave * steps * 64;
  int id[TABLE_STEPS];
#pragma unroll
  for (int s = 0; s < TABLE_STEPS; ++s) {
    const int i = first + s * 64 + lane;
    id[s] = s < steps && i < end_slot ? topk_ids[i] : -1;
  }
  int* const all = counts + TABLE_WAVES * num_experts;
  for (int i = tid; i < (alone ? 1 : 2) * TABLE_WAVES * num_experts; i += TABLE_THREADS) counts[i] = 0;
  __syncthreads();
  int* mine = counts + wave * num_experts;
#pragma unroll
  for (int s = 0; s < TABLE_STEPS; ++s) {
    if (s >= steps) break;
    if ((uint32_t)id[s] < (uint32_t)num_experts) atomicAdd(mine + id[s], 1);
  }
  if (!alone) {
    int* const mine_all = all + wave * num_experts;
#pragma unroll 8
    for (int i = tid; i < topk_length; i += TABLE_THREADS) {
      const int e = topk_ids[i];
      if ((uint32_t)e < (uint32_t)num_experts) atomicAdd(mine_all + e, i < begin_slot ? 65537 : 1);
    }
  }
  __syncthreads();
  // one thread per expert (num_experts <= 512): rows and tiles, then their running sums over the block
  int rows = 0, tiles = 0;
  if (tid < num_experts) {
    int before = 0;  // this expert's slots in earlier segments, then in earlier waves too
    if (!alone) {
#pragma unroll
      for (int w = 0; w < TABLE_WAVES; ++w) {
        const int c = all[w * num_experts + tid];
        rows += c & 0xffff;
        before += c >> 16;
      }
    }
#pragma unroll
    for (int w = 0; w < TABLE_WAVES; ++w) {
      const int c = counts[w * num_experts + tid];
      counts[w * num_experts + tid] = before;
      before += c;
    }
    if (alone) rows = before;
    tiles = (rows + plan_rows - 1) / plan_rows;
  }
  int row_sum = rows, tile_sum = tiles;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int r = __shfl_up(row_sum, d), t = __shfl_up(tile_sum, d);
    row_sum += lane >= d ? r : 0;
    tile_sum += lane >= d ? t : 0;
  }
  if (lane == 63) {
    wave_rows[wave] = row_sum;
    wave_tiles[wave] = tile_sum;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < TABLE_WAVES; ++w) {
    row_sum += w < wave ? wave_rows[w] : 0;
    tile_sum += w < wave ? wave_tiles[w] : 0;
  }
  if (tid < num_experts) {
    const int begin = row_sum - rows;
#pragma unroll
    for (int w = 0; w < TABLE_WAVES; ++w) counts[w * num_experts + tid] += begin;
    if (blockIdx.x == 0) {
      if (tid == 0) expert_offsets[0] = 0;
      expert_offsets[tid + 1] = row_sum;
      ps1[3 * tid] = rows;
      ps1[3 * tid + 1] = 2 * n;
      ps1[3 * tid + 2] = k;
      ps2[3 * tid] = rows;
      ps2[3 * tid + 1] = k;
      ps2[3 * tid + 2] = n;
      // (the layout grouped_plan_kernel writes: expert, first row, end row)
      for (int i = 0, slot = tile_sum - tiles; i < tiles && slot < plan_max_tiles; ++i, ++slot)
        reinterpret_cast<v4i*>(plan)[1 + slot] = v4i{tid, begin + i * plan_rows, row_sum, 0};
      if (tid == num_experts - 1) plan[0] = tile_sum < plan_max_tiles ? tile_sum : plan_max_tiles;
    }
    if ((int)blockIdx.x >= walks.first_block) {
      expert_rows[tid] = rows;
      expert_end[tid] = row_sum;
      expert_tiles[tid] = tile_sum;
    }
  }
  __syncthreads();
  if ((int)blockIdx.x >= walks.first_block) {
    const uint32_t all_tiles = (uint32_t)expert_tiles[num_experts - 1], units1 = all_tiles * walks.columns[0].d;
    const uint32_t units = units1 + all_tiles * walks.columns[1].d;
    if ((int)blockIdx.x == walks.first_block && tid < 2) walks.walk[tid][0] = (int)(tid == 0 ? units1 : units - units1);
    for (uint32_t i = (blockIdx.x - walks.first_block) * TABLE_THREADS + tid; i < units; i += (uint32_t)(quant.first_block - walks.first_block) * TABLE_THREADS) {
      const bool one = i < units1;
      const int columns = (int)(one ? walks.columns[0].d : walks.columns[1].d);
      const uint32_t u = one ? i : i - units1;
      const int any = (int)(one ? walks.columns[0].div(u) : walks.columns[1].div(u));  // a row tile of the unit's expert: their units follow each other
      int e = 0;  // ... the first expert whose tiles end behind it
      for (int step = 1 << (id_bits > 0 ? id_bits - 1 : 0); step > 0; step >>= 1)
        if (e + step <= num_experts && expert_tiles[e + step - 1] <= any) e += step;
      const int rows_e = expert_rows[e], end = expert_end[e];
      const int count = (rows_e + WALK_ROWS - 1) / WALK_ROWS, first = expert_tiles[e] - count;
      const int bands = (count + WALK_BAND - 1) / WALK_BAND, height = bands == 1 ? count : (count + bands - 1) / bands;
      const int unit = (int)u - first * columns, band = bands == 1 ? 0 : (any - first) / height;
      const int left = count - band * height, rows_b = left < height ? left : height;
      const int in_band = unit - band * height * columns, column = in_band / rows_b;
      const int t = band * height + in_band - column * rows_b;
      // an expert's last two tiles share the rows that are left: the first half of them, rounded up to 32, and the rest
      int row = end - rows_e + t * WALK_ROWS, to = end;
      const int rest = to - row;
      const bool second = rest <= WALK_ROWS && t > 0;
      const int both = second ? rest + WALK_ROWS : rest, share = ((both + 1) / 2 + 31) & ~31;
      if (second) row += share - WALK_ROWS;
      else if (rest > WALK_ROWS) to = row + (rest < 2 * WALK_ROWS ? share : WALK_ROWS);
      reinterpret_cast<v4i*>((one ? walks.walk[0] : walks.walk[1]) + WALK_HEADER)[u] = v4i{row, to, e, column};
    }
    return;
  }
  const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
  for (int s = 0; s < TABLE_STEPS; ++s) {
    if (s >= steps) break;
    const int e = id[s];
    const bool live = (uint32_t)e < (uint32_t)num_experts;
    uint64_t same = __ballot(live);
    for (int b = 0; b < id_bits; ++b) {
      const uint64_t set = __ballot((e >> b) & 1);
      same &= ((e >> b) & 1) ? set : ~set;
    }
    const int i = first + s * 64 + lane;
    int pos = -1;
    if (live) {
      const int rank = __popcll(same & below);
      pos = mine[e] + rank;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (live && (same & below) == 0) mine[e] += __popcll(same);  // (the wave's LDS operations run in this order)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (i < end_slot) output_permutation[i] = pos;
    if (input_permutation && live) input_permutation[pos] = (int)topk.div((uint32_t)i);
  }
}

// ---------------------------------------------------------------------------
// shuffle_rows (prepare_moe_input.cu:168-244): output[d] = input[dst2src_map[d]], rows of
// row_bytes bytes.  16-byte pieces when rows and pointers allow, 4-byte or single bytes
// otherwise; a linear walk over (row, piece) pairs, so short rows (the 224-byte scale rows)
// use the lanes as well as long ones.
// ---------------------------------------------------------------------------
template <typename PIECE>
__global__ __launch_bounds__(256) void shuffle_rows_kernel(const char* __restrict__ in, const int* __restrict__ map,
                                                           char* __restrict__ out, int64_t num_src_rows,
                                                           int64_t num_dst_rows, int64_t row_bytes) {
  const int64_t ppr = row_bytes / (int64_t)sizeof(PIECE);  // pieces per row
  const int64_t total = num_dst_rows * ppr;
  for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < total; id += (int64_t)gridDim.x * 256) {
    const int64_t d = id / ppr, c = id - d * ppr;
    const int64_t s = map[d];
    if (s < 0 || s >= num_src_rows) continue;  // a map entry that names no row: the destination row is left alone
    reinterpret_cast<PIECE*>(out + d * row_bytes)[c] = reinterpret_cast<const PIECE*>(in + s * row_bytes)[c];
  }
}

// ---------------------------------------------------------------------------
// silu_and_mul (sgl-kernel/csrc/elementwise/activation.cu:57-60,85-103, the flashinfer
// act_and_mul kernel it instantiates): out[t, j] = T(silu(x[t, j])) * x[t, d + j] with the
// product rounded to T again; silu(v) = v / (1 + expf(-v)) in fp32.  16 bytes per lane.
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(256) void silu_and_mul_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                           int64_t tokens, int64_t d) {
  const int64_t cpr = d >> 3;  // 8-element chunks per output row
  const int64_t total = tokens * cpr;
  for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < total; id += (int64_t)gridDim.x * 256) {
    const int64_t t = id / cpr, c = id - t * cpr;
    const v4u xv = *reinterpret_cast<const v4u*>(in + t * 2 * d + c * 8);
    const v4u yv = *reinterpret_cast<const v4u*>(in + t * 2 * d + d + c * 8);
    v4u o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t w = 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        w |= (uint32_t)silu_mul_16<DT>((uint16_t)(xv[q] >> (16 * h)), (uint16_t)(yv[q] >> (16 * h))) << (16 * h);
      }
      o[q] = w;
    }
    *reinterpret_cast<v4u*>(out + t * d + c * 8) = o;
  }
}

// Rows whose halves are not 16-byte aligned (d not a multiple of 8): one element per lane.
template <int DT>
__global__ __launch_bounds__(256) void silu_and_mul_scalar_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                                  int64_t tokens, int64_t d) {
  const int64_t total = tokens * d;
  for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < total; id += (int64_t)gridDim.x * 256) {
    const int64_t t = id / d, c = id - t * d;
    out[id] = silu_mul_16<DT>(in[t * 2 * d + c], in[t * 2 * d + d + c]);
  }
}

// ---------------------------------------------------------------------------
// apply_shuffle_mul_sum (prepare_moe_input.cu:258-392): output[i, :] = sum over j < topk of
// factors[i * topk + j] * input[permutation[i * topk + j], :], accumulated in fp32 in j order
// with one fused multiply-add per term (:293-295), rounded once to the 16-bit type.
// A lane owns 8 consecutive elements of one output row; lanes walk (row, chunk) pairs linearly,
// so rows of any length fill the waves.
// FACTOR = float: the factors as the router leaves them, rounded to the 16-bit type here instead of by
// a conversion kernel in front (one launch of a decode step's chain).
// ---------------------------------------------------------------------------
template <int DT, typename FACTOR = uint16_t>
__global__ __launch_bounds__(256) void shuffle_mul_sum_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out,
                                                              const int* __restrict__ perm,
                                                              const FACTOR* __restrict__ factors, int64_t m, int topk,
                                                              int64_t row, int64_t num_src_rows) {
  auto factor = [&](int64_t slot) -> float {
    if constexpr (std::is_same<FACTOR, float>::value) return to_f32_16<DT>(from_f32_16<DT>(factors[slot]));
    else return to_f32_16<DT>(factors[slot]);
  };
  const int64_t cpr = row >> 3;  // chunks per row
  const int64_t total = m * cpr;
  for (int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x; id < total; id += (int64_t)gridDim.x * 256) {
    const int64_t i = id / cpr, c = id - i * cpr;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // Eight slots at a time: their table entries, then their rows, are loaded together so that one
    // memory round trip covers eight terms; the sum still runs in slot order.  A slot that names
    // no row (routed to nobody, or past topk) reads row 0 and enters as 0 * 0, which leaves the
    // sum as it is (the sum is never -0: it starts from +0).
    for (int j0 = 0; j0 < topk; j0 += 8) {
      int64_t src[8];
      float f[8];
      bool ok[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int64_t slot = i * topk + (j0 + u < topk ? j0 + u : topk - 1);
        src[u] = perm[slot];
        f[u] = factors ? factor(slot) : 1.0f;
      }
      v4u v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        ok[u] = j0 + u < topk && src[u] >= 0 && src[u] < num_src_rows;
        v[u] = *reinterpret_cast<const v4u*>(in + (ok[u] ? src[u] : 0) * row + c * 8);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float fu = ok[u] ? f[u] : 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t w = ok[u] ? v[u][q] : 0u;
          acc[2 * q] = __builtin_fmaf(fu, to_f32_16<DT>((uint16_t)(w & 0xffffu)), acc[2 * q]);
          acc[2 * q + 1] = __builtin_fmaf(fu, to_f32_16<DT>((uint16_t)(w >> 16)), acc[2 * q + 1]);
        }
      }
    }
    v4u o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = (uint32_t)from_f32_16<DT>(acc[2 * q]) | ((uint32_t)from_f32_16<DT>(acc[2 * q + 1]) << 16);
    *reinterpret_cast<v4u*>(out + i * row + c * 8) = o;
  }
}

}  // namespace sglq

using namespace sglq;

extern "C" int sglq_prepare_moe_input(const int32_t* topk_ids, int32_t* expert_offsets, int32_t* blockscale_offsets,
                                      int32_t* problem_sizes1, int32_t* problem_sizes2, int32_t* input_permutation,
                                      int32_t* output_permutation, int64_t topk_length, int64_t topk, int64_t num_experts,
                                      int64_t n, int64_t k, void* stream) {
  const char* name = "prepare_moe_input";
  if (topk_length < 0 || topk <= 0 || num_experts < 0 || num_experts >= (1 << 20) || n < 0 || k < 0 ||
      n >= (1ll << 30) || k >= (1ll << 31) || topk_length >= (1ll << 31)) {
    set_error("%s: bad sizes", name);
    return SGLQ_EINVAL;
  }
  if (num_experts == 0) return SGLQ_OK;
  if (!expert_offsets || !problem_sizes1 || !problem_sizes2 || (topk_length > 0 && (!topk_ids || !input_permutation || !output_permutation))) {
    set_error("%s: null pointer", name);
    return SGLQ_EINVAL;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int aligned = (reinterpret_cast<uintptr_t>(topk_ids) & 15) == 0;
  moe_count_kernel<<<dim3((uint32_t)num_experts), dim3(MOE_THREADS), 0, st>>>(topk_ids, problem_sizes1, problem_sizes2, topk_length,
                                                                              (int)n, (int)k, aligned);
  moe_offsets_kernel<<<dim3(1), dim3(256), 0, st>>>(problem_sizes1, expert_offsets, blockscale_offsets, (int)num_experts);
  if (topk_length > 0) {
    // few experts: several blocks per expert, each with its own range of slots (about one block per CU in all)
    const int64_t sweeps = (topk_length + MOE_SWEEP - 1) / MOE_SWEEP;
    int64_t parts = 256 / num_experts;
    if (parts > sweeps) parts = sweeps;
    if (parts < 1) parts = 1;
    const int64_t span = (sweeps + parts - 1) / parts * MOE_SWEEP;
    moe_place_kernel<<<dim3((uint32_t)num_experts, (uint32_t)parts), dim3(MOE_THREADS), 0, st>>>(
        topk_ids, expert_offsets, input_permutation, output_permutation, topk_length, (int)topk, span, aligned);
  }
  return check_moe_launch(name);
}

static int prepare_layer_entry(const int32_t* topk_ids, int32_t* expert_offsets, int32_t* problem_sizes1, int32_t* problem_sizes2,
                               int32_t* output_permutation, int32_t* input_permutation, int64_t topk, int64_t topk_length,
                               int64_t num_experts, int64_t n, int64_t k, int64_t plan_rows, int64_t plan_max_tiles, void* plan, void* stream,
                               void* walk1 = nullptr, void* walk2 = nullptr, LayerQuant quant = LayerQuant{}, int quant_dtype = -1, bool once = false) {
  const char* name = "prepare_moe_layer";
  if (topk_length <= 0 || num_experts <= 0 || n < 0 || k < 0 || n >= (1ll << 30) || k >= (1ll << 31) || plan_rows <= 0 ||
      plan_max_tiles <= 0 || plan_max_tiles >= (1ll << 27) || topk <= 0 || topk >= (1 << 20)) {
    set_error("%s: bad sizes", name);
    return SGLQ_EINVAL;
  }
  if (topk_length > TABLE_MAX_SLOTS || num_experts > TABLE_MAX_EXPERTS) {
    set_error("%s: up to %d slots and %d experts (larger layers: sglq_prepare_moe_input)", name, TABLE_MAX_SLOTS, TABLE_MAX_EXPERTS);
    return SGLQ_EUNSUPPORTED;
  }
  if (!topk_ids || !expert_offsets || !problem_sizes1 || !problem_sizes2 || !output_permutation || !plan ||
      (reinterpret_cast<uintptr_t>(plan) & 15)) {
    set_error("%s: null pointer, or a plan that is not 16-byte aligned", name);
    return SGLQ_EINVAL;
  }
  int id_bits = 0;
  while ((1 << id_bits) < num_experts) ++id_bits;
  FastDiv per_token;
  per_token.init((uint32_t)topk);
  int64_t segments = 1;
  if (topk_length > TABLE_ONE_SEGMENT && num_experts <= TABLE_SEGMENTS_EXPERTS) segments = (topk_length + TABLE_SEGMENT - 1) / TABLE_SEGMENT;
  const int64_t segment = ((topk_length + segments - 1) / segments + TABLE_THREADS - 1) / TABLE_THREADS * TABLE_THREADS;
  segments = (topk_length + segment - 1) / segment;
  LayerWalks walks{};
  walks.first_block = (int)segments;
  int64_t walk_blocks = 0;
  if (walk1) {
    walks.walk[0] = static_cast<int*>(walk1);
    walks.walk[1] = static_cast<int*>(walk2);
    walks.columns[0].init((uint32_t)((2 * n + 255) / 256));
    walks.columns[1].init((uint32_t)((k + 255) / 256));
    walk_blocks = (plan_max_tiles * (walks.columns[0].d + walks.columns[1].d) + TABLE_THREADS - 1) / TABLE_THREADS;
    if (walk_blocks > 32) walk_blocks = 32;
  }
  const size_t lds = (size_t)(segments + walk_blocks > 1 ? 2 : 1) * TABLE_WAVES * num_experts * sizeof(int);
  quant.first_block = (int)(segments + walk_blocks);
  int64_t quant_blocks = 0;
  if (quant_dtype >= 0) {
    quant.walk.init((quant.groups_per_row + 8 * QUANT_WAVES - 1) / (8 * QUANT_WAVES));
    quant_blocks = (int64_t)((quant.num_tokens + QUANT_TOKENS - 1) / QUANT_TOKENS) * quant.walk.d;
  }
  const dim3 grid((uint32_t)(segments + walk_blocks + quant_blocks)), block(TABLE_THREADS);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define SGLQ_TABLES(DT, ONCE)                                                                                                                          \
  moe_tables_kernel<DT, ONCE><<<grid, block, lds, st>>>(topk_ids, expert_offsets, problem_sizes1, problem_sizes2, output_permutation,                 \
                                                        input_permutation, per_token, (int)topk_length, (int)num_experts, id_bits, (int)n, (int)k,    \
                                                        static_cast<int*>(plan), (int)plan_rows, (int)plan_max_tiles, (int)segment, walks, quant)
  if (quant_dtype == SGLQ_BF16 && once) SGLQ_TABLES(SGLQ_BF16, true);
  else if (quant_dtype == SGLQ_BF16) SGLQ_TABLES(SGLQ_BF16, false);
  else if (quant_dtype == SGLQ_FP16 && once) SGLQ_TABLES(SGLQ_FP16, true);
  else if (quant_dtype == SGLQ_FP16) SGLQ_TABLES(SGLQ_FP16, false);
  else SGLQ_TABLES(-1, false);
#undef SGLQ_TABLES
  return check_moe_launch(name);
}

extern "C" int sglq_prepare_moe_layer(const int32_t* topk_ids, int32_t* expert_offsets, int32_t* problem_sizes1,
                                      int32_t* problem_sizes2, int32_t* output_permutation, int64_t topk_length,
                                      int64_t num_experts, int64_t n, int64_t k, int64_t plan_rows, int64_t plan_max_tiles,
                                      void* plan, void* stream) {
  return prepare_layer_entry(topk_ids, expert_offsets, problem_sizes1, problem_sizes2, output_permutation, nullptr, 1, topk_length, num_experts, n, k,
                             plan_rows, plan_max_tiles, plan, stream);
}

extern "C" int sglq_prepare_moe_layer_rows(const int32_t* topk_ids, int32_t* expert_offsets, int32_t* problem_sizes1,
                                           int32_t* problem_sizes2, int32_t* output_permutation, int32_t* input_permutation,
                                           int64_t topk, int64_t topk_length, int64_t num_experts, int64_t n, int64_t k,
                                           int64_t plan_rows, int64_t plan_max_tiles, void* plan, void* stream) {
  if (!input_permutation) {
    set_error("prepare_moe_layer_rows: null pointer");
    return SGLQ_EINVAL;
  }
  return prepare_layer_entry(topk_ids, expert_offsets, problem_sizes1, problem_sizes2, output_permutation, input_permutation, topk, topk_length,
                             num_experts, n, k, plan_rows, plan_max_tiles, plan, stream);
}

extern "C" int sglq_prepare_moe_layer_walks(const int32_t* topk_ids, int32_t* expert_offsets, int32_t* problem_sizes1, int32_t* problem_sizes2,
                                            int32_t* output_permutation, int32_t* input_permutation, int64_t topk, int64_t topk_length,
                                            int64_t num_experts, int64_t n, int64_t k, void* plan, void* walks, int64_t walks_bytes, void* stream) {
  int64_t second = 0;
  const int64_t need = sglq_grouped_walk_bytes(num_experts, topk_length, n, k, &second);
  if (!input_permutation || !walks || (reinterpret_cast<uintptr_t>(walks) & 15) || need == 0 || walks_bytes < need) {
    set_error("prepare_moe_layer_walks: a row map and 16-byte aligned walks of %lld bytes are needed, for sizes that sglq_grouped_walk_bytes names", (long long)need);
    return SGLQ_EINVAL;
  }
  return prepare_layer_entry(topk_ids, expert_offsets, problem_sizes1, problem_sizes2, output_permutation, input_permutation, topk, topk_length,
                             num_experts, n, k, WALK_ROWS, topk_length / WALK_ROWS + num_experts, plan, stream, walks, static_cast<char*>(walks) + second);
}

extern "C" int sglq_prepare_moe_layer_quant(const int32_t* topk_ids, int32_t* expert_offsets, int32_t* problem_sizes1, int32_t* problem_sizes2,
                                            int32_t* output_permutation, int32_t* input_permutation, int64_t topk, int64_t topk_length,
                                            int64_t num_experts, int64_t n, int64_t k, int64_t plan_rows, int64_t plan_max_tiles, void* plan,
                                            void* walks, int64_t walks_bytes, const void* input, int in_dtype, void* output_q, float* output_s,
                                            int once, float eps, void* stream) {
  const char* name = "prepare_moe_layer_quant";
  if (topk <= 0 || topk > QUANT_MAX_TOPK || topk_length <= 0 || topk_length > QUANT_MAX_SLOTS || topk_length % topk != 0 || k <= 0 || k % 128 != 0) {
    set_error("%s: up to %d slots, %d a token, k (%lld) a multiple of 128", name, QUANT_MAX_SLOTS, QUANT_MAX_TOPK, (long long)k);
    return SGLQ_EINVAL;
  }
  if (in_dtype != SGLQ_BF16 && in_dtype != SGLQ_FP16) {
    set_error("%s: unsupported in_dtype %d", name, in_dtype);
    return SGLQ_EUNSUPPORTED;
  }
  if (!input || !output_q || !output_s || (reinterpret_cast<uintptr_t>(input) & 15) || (reinterpret_cast<uintptr_t>(output_q) & 7) || !(eps > 0.f)) {
    set_error("%s: input must be 16-byte and output_q 8-byte aligned, eps positive", name);
    return SGLQ_EINVAL;
  }
  int64_t second = 0;
  if (walks && (plan_rows != WALK_ROWS || plan_max_tiles != topk_length / WALK_ROWS + num_experts || !input_permutation || (reinterpret_cast<uintptr_t>(walks) & 15) ||
                sglq_grouped_walk_bytes(num_experts, topk_length, n, k, &second) == 0 ||
                walks_bytes < sglq_grouped_walk_bytes(num_experts, topk_length, n, k, &second))) {
    set_error("%s: walks need 256-row tiles, a row map and sglq_grouped_walk_bytes bytes, 16-byte aligned", name);
    return SGLQ_EINVAL;
  }
  LayerQuant quant{};
  quant.x = static_cast<const char*>(input);
  quant.q = static_cast<char*>(output_q);
  quant.s = output_s;
  quant.num_tokens = (uint32_t)(topk_length / topk);
  quant.groups_per_row = (uint32_t)(k / 128);
  quant.eps = eps;
  quant.qmax = 448.0f;
  quant.rqmax = 1.0f / 448.0f;
  return prepare_layer_entry(topk_ids, expert_offsets, problem_sizes1, problem_sizes2, output_permutation, input_permutation, topk, topk_length, num_experts, n, k,
                             plan_rows, plan_max_tiles, plan, stream, walks, walks ? static_cast<char*>(walks) + second : nullptr, quant, in_dtype, once != 0);
}

extern "C" int sglq_shuffle_rows(const void* input, const int32_t* dst2src_map, void* output, int64_t num_src_rows,
                                 int64_t num_dst_rows, int64_t row_bytes, void* stream) {
  const char* name = "shuffle_rows";
  if (num_src_rows < 0 || num_dst_rows < 0 || row_bytes < 0) {
    set_error("%s: negative size", name);
    return SGLQ_EINVAL;
  }
  if (num_dst_rows == 0 || row_bytes == 0) return SGLQ_OK;
  if (!input || !dst2src_map || !output) {
    set_error("%s: null pointer", name);
    return SGLQ_EINVAL;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const char* in = static_cast<const char*>(input);
  char* out = static_cast<char*>(output);
  const uintptr_t align = reinterpret_cast<uintptr_t>(input) | reinterpret_cast<uintptr_t>(output) | (uintptr_t)row_bytes;
  const int piece = (align & 15) == 0 ? 16 : (align & 3) == 0 ? 4 : 1;
  const int64_t total = num_dst_rows * (row_bytes / piece);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  const dim3 grid((uint32_t)blocks), block(256);
  if (piece == 16) shuffle_rows_kernel<v4u><<<grid, block, 0, st>>>(in, dst2src_map, out, num_src_rows, num_dst_rows, row_bytes);
  else if (piece == 4) shuffle_rows_kernel<uint32_t><<<grid, block, 0, st>>>(in, dst2src_map, out, num_src_rows, num_dst_rows, row_bytes);
  else shuffle_rows_kernel<unsigned char><<<grid, block, 0, st>>>(in, dst2src_map, out, num_src_rows, num_dst_rows, row_bytes);
  return check_moe_launch(name);
}

extern "C" int sglq_silu_and_mul(const void* input, int dtype, void* output, int64_t num_tokens, int64_t d, void* stream) {
  const char* name = "silu_and_mul";
  if (num_tokens < 0 || d < 0) {
    set_error("%s: negative size", name);
    return SGLQ_EINVAL;
  }
  if (num_tokens == 0 || d == 0) return SGLQ_OK;
  if (!input || !output) {
    set_error("%s: null pointer", name);
    return SGLQ_EINVAL;
  }
  if (dtype != SGLQ_BF16 && dtype != SGLQ_FP16) {
    set_error("%s: dtype must be Half or BFloat16", name);
    return SGLQ_EUNSUPPORTED;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool wide = d % 8 == 0 && !(reinterpret_cast<uintptr_t>(input) & 15) && !(reinterpret_cast<uintptr_t>(output) & 15);
  const int64_t total = wide ? num_tokens * (d / 8) : num_tokens * d;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  const dim3 grid((uint32_t)blocks), block(256);
  const uint16_t* in = static_cast<const uint16_t*>(input);
  uint16_t* out = static_cast<uint16_t*>(output);
  if (wide) {
    if (dtype == SGLQ_BF16) silu_and_mul_kernel<SGLQ_BF16><<<grid, block, 0, st>>>(in, out, num_tokens, d);
    else silu_and_mul_kernel<SGLQ_FP16><<<grid, block, 0, st>>>(in, out, num_tokens, d);
  } else {
    if (dtype == SGLQ_BF16) silu_and_mul_scalar_kernel<SGLQ_BF16><<<grid, block, 0, st>>>(in, out, num_tokens, d);
    else silu_and_mul_scalar_kernel<SGLQ_FP16><<<grid, block, 0, st>>>(in, out, num_tokens, d);
  }
  return check_moe_launch(name);
}

static int shuffle_mul_sum_entry(const void* input, void* output, const int32_t* permutation, const void* factors, bool f32_factors,
                                 int dtype, int64_t m, int64_t topk, int64_t row, int64_t num_src_rows, void* stream) {
  const char* name = "apply_shuffle_mul_sum";
  if (m < 0 || topk <= 0 || row < 0 || num_src_rows < 0 || topk >= (1 << 20) || m >= (1ll << 31)) {
    set_error("%s: bad sizes", name);
    return SGLQ_EINVAL;
  }
  if (m == 0 || row == 0) return SGLQ_OK;
  if (num_src_rows == 0) {
    set_error("%s: input has no rows", name);
    return SGLQ_EINVAL;
  }
  if (!input || !output || !permutation) {
    set_error("%s: null pointer", name);
    return SGLQ_EINVAL;
  }
  if (row % 8 != 0 || (reinterpret_cast<uintptr_t>(input) & 15) || (reinterpret_cast<uintptr_t>(output) & 15)) {
    set_error("%s: rows must be multiples of 8 elements and 16-byte aligned", name);
    return SGLQ_EINVAL;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  int64_t blocks = (m * (row / 8) + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  const dim3 grid((uint32_t)blocks), block(256);
  const uint16_t* in = static_cast<const uint16_t*>(input);
  uint16_t* out = static_cast<uint16_t*>(output);
#define SGLQ_COMBINE(DT, F)                                                                                                   \
  shuffle_mul_sum_kernel<DT, F><<<grid, block, 0, st>>>(in, out, permutation, static_cast<const F*>(factors), m, (int)topk, row, \
                                                        num_src_rows)
  if (dtype == SGLQ_BF16 && f32_factors) SGLQ_COMBINE(SGLQ_BF16, float);
  else if (dtype == SGLQ_BF16) SGLQ_COMBINE(SGLQ_BF16, uint16_t);
  else if (dtype == SGLQ_FP16 && f32_factors) SGLQ_COMBINE(SGLQ_FP16, float);
  else if (dtype == SGLQ_FP16) SGLQ_COMBINE(SGLQ_FP16, uint16_t);
#undef SGLQ_COMBINE
  else {
    set_error("%s: dtype must be Half or BFloat16", name);
    return SGLQ_EUNSUPPORTED;
  }
  return check_moe_launch(name);
}

extern "C" int sglq_apply_shuffle_mul_sum(const void* input, void* output, const int32_t* permutation, const void* factors,
                                          int dtype, int64_t m, int64_t topk, int64_t row, int64_t num_src_rows,
                                          void* stream) {
  return shuffle_mul_sum_entry(input, output, permutation, factors, false, dtype, m, topk, row, num_src_rows, stream);
}

extern "C" int sglq_apply_shuffle_mul_sum_f32(const void* input, void* output, const int32_t* permutation, const float* factors,
                                              int dtype, int64_t m, int64_t topk, int64_t row, int64_t num_src_rows,
                                              void* stream) {
  return shuffle_mul_sum_entry(input, output, permutation, factors, true, dtype, m, topk, row, num_src_rows, stream);
}
