// Device pieces that the GEMM translation units share: the problem description, the global -> LDS copies,
// the operand layout and the scale-and-store epilogues (the layout of the computation is described at the
// head of gemm.hip).
#pragma once
#include <type_traits>
#include <utility>

#include "sglq_common.h"

namespace sglq {

// f(0), f(1) ... f(N - 1), each with its index as a constant
template <int... I, typename F>
SGLQ_DEV void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
SGLQ_DEV void static_for(F&& f) {
  static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

constexpr int KIND_FP8_BLOCK = 0;   // a4: sum_kb P_kb * sfa[m,kb] * sfb[kb,n/128]
constexpr int KIND_FP8_ROWCOL = 1;  // a6: sa[m] * (sb[n] * acc) + bias[n]
constexpr int KIND_I8_ROWCOL = 2;   // a5: float(acc) * (sb[n] * sa[m]) + bias[n]
constexpr int KIND_I8_RAW = 3;      // INT32 accumulators
constexpr int KIND_I8_BLOCK = 4;    // block-scaled INT8: sum_kb float(P_kb) * sfa[m,kb] * sfb[kb,n/128]
// KIND_FP8_BLOCK whose scales are all powers of two (UE8M0 values held as fp32): the MFMA applies them itself
// (v_mfma_scale_f32_16x16x128_f8f6f4 takes an exponent byte per lane for each operand) and accumulates in place,
// so there is no scale-and-accumulate pass behind every MFMA.  The 256- and 128-row pipelined kernels and, above 128
// rows, gemm_ring_kernel are built for it; everywhere else such scales run as KIND_FP8_BLOCK (the same sums folded per K block: equal to the
// in-place accumulation up to the order of the additions, not bit for bit).
constexpr int KIND_FP8_BLOCK_POW2 = 5;

constexpr bool is_block(int kind) { return kind == KIND_FP8_BLOCK || kind == KIND_I8_BLOCK || kind == KIND_FP8_BLOCK_POW2; }
constexpr bool fp8_operands(int kind) { return kind == KIND_FP8_BLOCK || kind == KIND_FP8_ROWCOL || kind == KIND_FP8_BLOCK_POW2; }
// the biased exponent of a positive power of two = its UE8M0 code, in byte 0 as the scaled MFMA reads it
SGLQ_DEV int ue8m0_of(float pow2) { return (int)(__builtin_bit_cast(uint32_t, pow2) >> 23); }
// ... of an activation scale as the kernels hold it: the eight bits from `shift` on, 23 for an fp32 power of two, 8 (kb % 4)
// for a word of four UE8M0 codes (GemmArgs::sa_packed) and K block kb
SGLQ_DEV int ue8m0_at(float word, int shift) { return (int)((__builtin_bit_cast(uint32_t, word) >> shift) & 0xffu); }
constexpr bool float_acc(int kind) { return fp8_operands(kind) || kind == KIND_I8_BLOCK; }

constexpr uint32_t OOB = 0x80000000u;  // offset beyond any buffer this library accepts
constexpr uint32_t SC_NONE = 0x40000000u;  // scalar offset beyond any scale tensor (at most 2^31 / 32 bytes)

struct GemmArgs {
  const char* a;   // [M, K] bytes, row stride lda
  const char* b;   // [N, K] bytes, row stride ldb (column-major [K, N])
  const float* sa; // block: sfa; rowcol: scales_a [M]
  const float* sb; // block: sfb; rowcol: scales_b [N]
  const void* bias;
  void* out;
  int64_t sa_stride_m, sa_stride_k;  // block scales
  int64_t sb_stride_k, sb_stride_n;
  int64_t ldo;
  uint32_t lda, ldb;
  uint32_t a_bytes, b_bytes;
  int M, N, K;
  int tiles_m, tiles_n;
  void* ws;        // split-K partial sums [splits][M][N], fp32 or int32; grouped GEMM: the tile plan
  int splits;
  int64_t b_expert_stride, sb_expert_stride;  // grouped GEMM: bytes / floats between experts' weights / weight scales
  int num_experts;
  float* out_scales;   // grouped GEMM with the activation behind it (PIPE_SILU): scales of its FP8 outputs, [N / 256][M]
  const int* walk;     // grouped GEMM on 256-row tiles: its walk (nullptr: in the order of the plan)
  const int* row_map;  // grouped GEMM: row m of A is row row_map[m] of `a`, which has map_rows rows (nullptr: row m)
  int map_rows;
  int stream_out;  // the output is larger than the last-level cache: store it with the non-temporal hint
  int pow2_scales;  // block-scaled FP8: every scale is a power of two (KIND_FP8_BLOCK_POW2 where it is built)
  // ... and the activation scales come as UE8M0 codes, four K blocks to an int32 word: word (m, kb / 4) sits at
  // sa[m * sa_stride_m + (kb / 4) * sa_stride_k], byte kb % 4 of it is K block kb's code (what
  // sglq_per_token_group_quant_fp8_ue8m0 writes).  Read as they are by the KIND_FP8_BLOCK_POW2 kernels; every
  // other kernel gets them expanded to fp32 first (expand_packed_scales).
  int sa_packed;
  float* sa_expanded;  // room for [M, K / 128] fp32 scales (sa_packed only)
  float quant_eps;  // fused quantization (gemm_stream_quant_kernel): lower bound of a group's abs-max
  int cus;          // compute units of the call's device (host: the choice of a kernel and its grid)
};

// Where a tile of weight rows starts its way round K (of `steps` steps).  With weight rows a multiple of 4 KiB apart a K
// block of every row lies in the same few memory channels, and blocks that start together walk K in step, so they are
// bound by those channels instead of the memory; each tile starts at a place of its own instead (the golden ratio spreads
// neighbours).  A plain copy in gemm_stream_kernel's order shows the same: 28672 x 4096 in blocks of 16 rows 22.0 us in step, 20.5 us so,
// of 32 rows 23.2 and 20.8.
// On that kernel, weights rotated through more than the last-level cache, 1 and 16 rows, before and after: 28672 x 4096
// 25.7 -> 23.2 and 27.0 -> 24.4 us, 8192 x 4096 9.9 -> 8.7 and 10.2 -> 8.9, 4096 x 4096 5.8 -> 5.2 and 6.0 -> 5.4,
// 7168 x 16384 26.2 -> 23.9 and 28.0 -> 26.2, 57344 x 8192 80.9 -> 78.5 and 92.8 -> 90.9; nothing on rows of 1, 2, 6, 7
// or 14 KiB, which stay in order.
// Grouped (gemm_kernel, gemm_ring_kernel): the tile is one of all experts' weights, and row tiles of one expert start together; whatever the rows, since an
// expert's are few where these kernels run.  Layers in step and so, us: 64 x 8, 4096 x 1024 8 / 64 / 256 tokens 122 / 185 / 231 -> 105 / 161 / 212; 16 x 4, 4096 x 2048
// 16 / 64 / 128 tokens 102 / 118 / 148 -> 85 / 102 / 100; 32 x 8, 8192 x 2048 32 / 64 / 256 tokens 308 / 392 / 384 -> 303 / 320 / 366; 32 x 4, 4096 x 4096 8 / 176
// tokens 169 / 362 -> 148 / 315.  Weights that the last-level cache holds: even (8 x 2, 4096 x 2048 50.1 -> 51.1 at worst).
SGLQ_DEV int first_k_step(const GemmArgs& p, uint32_t tile, int steps) {
  if (p.ldb & 4095) return 0;
  return (int)(((tile * 40503u & 0xffffu) * (uint32_t)steps) >> 16);  // 40503 / 2^16: the golden ratio
}
// The number of a grouped tile of 128 weight rows.  Where N is two halves of whole tiles, gates and their partners, a tile has the number of the other half's: gemm_few_rows_kernel's
// tiles are 128 rows of each, start once, and so sum in the GEMM's order.  (A number of its own for every tile is no faster: 70 layers on such weights 1.000 of the time on average, 0.977 to 1.027.)
SGLQ_DEV uint32_t grouped_weight_tile(const GemmArgs& p, int expert, int tn) {
  const int half = p.N & 255 ? (p.N + 127) >> 7 : p.N >> 8;
  return (uint32_t)(expert * half + (tn < half ? tn : tn - half));
}
// ... for kernels whose blocks also share an activation tile, which in step they read from their L2 together: only where
// the weights are what is read (48 weight rows to an activation row) and the activations stay in the L2 anyway (2 MiB).
// gemm_ring_kernel, in step and so: 24 x 28672 x 4096 30.6 -> 24.4 us, 64 x 57344 x 8192 107 -> 88, 200 x 14336 x 4096
// 25.0 -> 22.5, 64 x 8192 x 8192 21.6 -> 19.9; gemm_kwave_kernel: 32 x 14336 x 4096 16.5 -> 14.7, 96 x 28672 x 4096
// 33.5 -> 29.2; gemm_skinny_kernel without split-K: 64 x 14336 x 4096 18.2 -> 16.1 (with it the splits of a weight tile
// read neighbouring K blocks already: 40 x 5120 x 8192 16.5 -> 17.7 us, left in step).  Past the bounds it loses:
// 230 x 6144 x 8192 27.1 -> 29.6 us, 512 x 10240 x 8192 51.2 -> 54.7, 333 x 7168 x 16384 66.7 -> 84.1; another start for
// each XCD there is no gain either (1024 x 7168 x 16384 119.8 -> 117.8, but 333 rows 66.7 -> 69.2).
static __host__ __device__ __forceinline__ bool spreads_k_starts(const GemmArgs& p) {
  return !(p.ldb & 4095) && 48 * (int64_t)p.M <= p.N && p.a_bytes <= 2u << 20;
}
SGLQ_DEV int first_k_step_shared(const GemmArgs& p, uint32_t tile, int steps) { return spreads_k_starts(p) ? first_k_step(p, tile, steps) : 0; }

// Grouped GEMM tile plan in the workspace (int32): [0] = number of row tiles, then from [4] on
// one entry of four per row tile: expert, first row, end row (both absolute rows of A and C).
constexpr int PLAN_HEADER = 4, PLAN_ENTRY = 4;

// Walk of a grouped GEMM on 256-row tiles (int32, sglq_prepare_moe_layer_walks): [0] = number of tiles, then from [WALK_HEADER] on one entry of four per
// tile, in the order in which they are taken: first row, end row (at most 256 rows on; where it is fewer, the tile computes only these), expert, column tile.
constexpr int WALK_HEADER = 16;

// s_waitcnt immediate: wait until at most `vm` vector-memory loads are outstanding
// and all LDS / scalar-memory operations are done (vmcnt is split over bits 3:0 and 15:14).
constexpr int waitcnt_vm_lgkm0(int vm) { return (vm & 0xf) | (((vm >> 4) & 3) << 14) | (7 << 4); }
// ... and one that waits for LDS / scalar-memory operations only
// Tile rows per band of the tile walk (tile_of_block).  Measured with the profiler's FETCH_SIZE counter (bytes
// that miss the XCDs' L2s) on the 256-row kernels at M = 4096: bands of 4 rows fetch 6 % less than bands of 8
// on 7168 x 16384 (224-wide tiles) and 20 % less on 2112 x 7168 (192-wide tiles), the same on 24576 x 1536 and
// 4096 x 7168 (with 32 tiles in flight per XCD, 4 x 8 and 8 x 4 touch the same number of rows when the tile is
// square); bands of 16 fetch 40-70 % more.  Launch times move by less than 2 % between 4 and 8 and by +2-3 %
// with 16: these kernels are not bound by that traffic.
#ifndef SGLQ_GROUP_M
#define SGLQ_GROUP_M 4
#endif
#ifndef SGLQ_STREAM_NSTAGE
#define SGLQ_STREAM_NSTAGE 3
#endif
constexpr int waitcnt_lgkm0_only() { return 0xf | (3 << 14) | (7 << 4); }

// Global -> LDS copies written as assembly (16 or 4 bytes per lane; lane l lands at
// lds_dst + l * size).  The decode kernel keeps several stages of such copies in flight and
// waits for them with explicit vmcnt counts; copies issued through the compiler's builtin
// are tracked by its wait-count pass, which cannot tell the ring's stages apart and would
// drain every copy in flight before each LDS read.
SGLQ_DEV v4u make_rsrc_sgpr(const void* ptr, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(ptr);
  return v4u{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
             (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
             (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
SGLQ_DEV void lds_copy16(v4u rsrc, uint32_t lds_dst, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(lds_dst), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
SGLQ_DEV void lds_copy4(v4u rsrc, uint32_t lds_dst, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds" : : "s"(lds_dst), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
SGLQ_DEV uint32_t lds_addr(const void* p) {
  return (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)p);
}

SGLQ_DEV int swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// One 128-byte K block of a block-scaled kind: the product of a weight and an activation
// fragment from a zero accumulator.  FP8: one MFMA, fp32 result.  INT8: two MFMAs, exact
// int32 result, returned as its bit pattern so that the conversion to float can wait until
// the result is folded into the accumulator (block_value) instead of stalling on the MFMA.
template <int KIND>
SGLQ_DEV v4f block_mfma(const v8i& w, const v8i& a) {
  if constexpr (KIND == KIND_I8_BLOCK) {
    const v4i w0 = {w[0], w[1], w[2], w[3]}, w1 = {w[4], w[5], w[6], w[7]};
    const v4i a0 = {a[0], a[1], a[2], a[3]}, a1 = {a[4], a[5], a[6], a[7]};
    v4i t = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, a0, v4i{0, 0, 0, 0}, 0, 0, 0);
    t = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, a1, t, 0, 0, 0);
    return __builtin_bit_cast(v4f, t);
  } else {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, a, v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
  }
}
template <int KIND>
SGLQ_DEV float block_value(float raw) {
  if constexpr (KIND == KIND_I8_BLOCK) return (float)__builtin_bit_cast(int, raw);
  else return raw;
}

template <int OUT_DT>
SGLQ_DEV void store4(void* out, int64_t idx, float v0, float v1, float v2, float v3) {
  if constexpr (OUT_DT == SGLQ_BF16) {
    typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
    bf4 o = {(__bf16)v0, (__bf16)v1, (__bf16)v2, (__bf16)v3};
    *reinterpret_cast<bf4*>(reinterpret_cast<__bf16*>(out) + idx) = o;
  } else {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    h4 o = {(_Float16)v0, (_Float16)v1, (_Float16)v2, (_Float16)v3};
    *reinterpret_cast<h4*>(reinterpret_cast<_Float16*>(out) + idx) = o;
  }
}

// fp32 -> output type -> fp32
template <int OUT_DT>
SGLQ_DEV float round_out(float v) {
  if constexpr (OUT_DT == SGLQ_BF16) return (float)(__bf16)v;
  else return (float)(_Float16)v;
}

template <int OUT_DT>
SGLQ_DEV void load_bias4(const void* bias, int n, float (&b)[4]) {
  if constexpr (OUT_DT == SGLQ_BF16) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(bias) + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = u2f((uint32_t)p[j] << 16);
  } else {
    const _Float16* p = reinterpret_cast<const _Float16*>(bias) + n;
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = (float)p[j];
  }
}

// Map the linear block id to an output tile: consecutive ids are dealt round-robin
// to the 8 XCDs by the dispatcher, so give every XCD one contiguous range of tiles
// (its L2 then sees a compact set of A rows and B columns), and walk each range in
// bands of GROUP_M tile-rows.
SGLQ_DEV void tile_of_block(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  const int q = total >> 3, rem = total & 7;
  const int xcd = pid & 7, idx = pid >> 3;
  int tile = xcd * q + (xcd < rem ? xcd : rem) + idx;
  constexpr int GROUP_M = SGLQ_GROUP_M;
  const int width = GROUP_M * tiles_n;
  const int group = tile / width;
  const int first_m = group * GROUP_M;
  const int gsz = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_group = tile - group * width;
  tm = first_m + in_group % gsz;
  tn = in_group / gsz;
}

// Scale, add bias and store four consecutive outputs C[m][n..n+3] from their accumulators.
// BLOCK_BIAS (block-scaled kinds only): 1 / 0 = the caller knows at compile time that there
// is / is not a bias, -1 = look at p.bias.
template <int KIND, int OUT_DT, int BLOCK_BIAS = -1, typename acc_t>
SGLQ_DEV void finish4(const GemmArgs& p, int m, int n, const acc_t& a, float sam) {
  const int64_t idx = (int64_t)m * p.ldo + n;
  if constexpr (KIND == KIND_I8_RAW) {
    *reinterpret_cast<v4i*>(reinterpret_cast<int32_t*>(p.out) + idx) = a;
  } else if constexpr (is_block(KIND)) {
    if (BLOCK_BIAS == 1 || (BLOCK_BIAS == -1 && p.bias)) {
      // the caller's `output += bias` on the rounded GEMM result (fp8_utils.py:210-211), fused:
      // round to the output type, add the bias in fp32, round again
      float bv[4], o[4];
      load_bias4<OUT_DT>(p.bias, n, bv);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = round_out<OUT_DT>(a[e]) + bv[e];
      store4<OUT_DT>(p.out, idx, o[0], o[1], o[2], o[3]);
    } else {
      store4<OUT_DT>(p.out, idx, a[0], a[1], a[2], a[3]);
    }
  } else {
    float o[4], bv[4] = {0.f, 0.f, 0.f, 0.f};
    const v4f sbn = *reinterpret_cast<const v4f*>(p.sb + n);
    if (p.bias) load_bias4<OUT_DT>(p.bias, n, bv);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (KIND == KIND_I8_ROWCOL) o[e] = __builtin_fmaf((float)a[e], sbn[e] * sam, bv[e]);
      else o[e] = __builtin_fmaf(sam, sbn[e] * a[e], bv[e]);
    }
    store4<OUT_DT>(p.out, idx, o[0], o[1], o[2], o[3]);
  }
}

// Split-K: store a wave's raw accumulators as partial sums of split `split` in the
// workspace, laid out [split][M][N] (fp32 or int32); splitk_reduce_kernel finishes them.
template <int MI, int NI, typename acc_t>
SGLQ_DEV void store_partials(const GemmArgs& p, acc_t (&acc)[MI][NI], int split, int m_base, int n_base, int r16, int g) {
  asm volatile("" : "+v"(r16), "+v"(g));  // keep the address arithmetic here (see epilogue_via_lds)
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m_base + i * 16 + r16;
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n_base + j * 16 + g * 4;
      if (n >= p.N) continue;
      acc_t* dst = reinterpret_cast<acc_t*>(reinterpret_cast<char*>(p.ws) + (((int64_t)split * p.M + m) * p.N + n) * 4);
      *dst = acc[i][j];
    }
  }
}

// The same for the 256-row kernels, as buffer stores that need neither branches nor 64-bit
// addresses: a row beyond M lies beyond the split's extent and is dropped by the bounds
// check, a column beyond N gets an offset that is.  The host keeps (M + 256) N 4 below 2 GiB.
template <int MI, int NI, typename acc_t>
SGLQ_DEV void store_partials_bounded(const GemmArgs& p, acc_t (&acc)[MI][NI], int split, int m_base, int n_base, int r16, int g) {
  asm volatile("" : "+v"(r16), "+v"(g));  // keep the address arithmetic here (see epilogue_via_lds)
  const uint32_t row_bytes = (uint32_t)p.N * 4u, split_bytes = (uint32_t)p.M * row_bytes;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(reinterpret_cast<char*>(p.ws) + (int64_t)split * split_bytes, split_bytes);
  const int n_lane = n_base + g * 4;
  const uint32_t off = (uint32_t)(m_base + r16) * row_bytes + (uint32_t)n_lane * 4u;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const uint32_t voff = (n_lane + j * 16 < p.N) ? off + (uint32_t)(i * 16) * row_bytes + (uint32_t)(j * 64) : OOB;
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, acc[i][j]), rw, voff, 0, 0);
    }
  }
}

// Scale, add bias and store a wave's accumulators.  acc[i][j][e] belongs to
// C[m_base + 16 i + r16][n_base + 16 j + 4 g + e].
template <int KIND, int OUT_DT, int MI, int NI, int BLOCK_BIAS = -1, typename acc_t>
SGLQ_DEV void epilogue(const GemmArgs& p, acc_t (&acc)[MI][NI], int m_base, int n_base, int r16, int g) {
  asm volatile("" : "+v"(r16), "+v"(g));  // keep the address arithmetic here (see epilogue_via_lds)
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m_base + i * 16 + r16;
    if (m >= p.M) continue;
    float sam = 1.f;
    if constexpr (KIND == KIND_FP8_ROWCOL || KIND == KIND_I8_ROWCOL) sam = p.sa[m];
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n_base + j * 16 + g * 4;
      if (n >= p.N) continue;  // N % 8 == 0 (% 4 for 32-bit outputs) is checked on the host: a run of 4 is in or out as a whole
      finish4<KIND, OUT_DT, BLOCK_BIAS>(p, m, n, acc[i][j], sam);
    }
  }
}

}  // namespace sglq
