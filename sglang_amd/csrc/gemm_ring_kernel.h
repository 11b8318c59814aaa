// gemm_ring_kernel (see gemm_ring.h) and its launcher for one kind.
#pragma once
#include "gemm_ring.h"

namespace sglq {

constexpr int RING_THREADS = 12 * 64;  // eight consumer and four producer waves

// Four consecutive outputs C[m][n .. n + 3] from their accumulators, before the final rounding.
template <int KIND, int OUT_DT, typename acc_t>
SGLQ_DEV void values4(const GemmArgs& p, int n, const acc_t& a, float sam, float (&o)[4]) {
  float bv[4] = {0.f, 0.f, 0.f, 0.f};
  if constexpr (is_block(KIND)) {
    if (p.bias) {
      load_bias4<OUT_DT>(p.bias, n, bv);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = round_out<OUT_DT>(a[e]) + bv[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = a[e];
    }
  } else {
    const v4f sbn = *reinterpret_cast<const v4f*>(p.sb + n);
    if (p.bias) load_bias4<OUT_DT>(p.bias, n, bv);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (KIND == KIND_I8_ROWCOL) o[e] = __builtin_fmaf((float)a[e], sbn[e] * sam, bv[e]);
      else o[e] = __builtin_fmaf(sam, sbn[e] * a[e], bv[e]);
    }
  }
}

// GROUPED: the row tiles, their experts and their last rows come from the plan in the workspace (see gemm_kernel).
template <int KIND, int OUT_DT, int WM, int WN, int KG, int MI, int NI, int NST, bool GROUPED = false>
__global__ __launch_bounds__(RING_THREADS) void gemm_ring_kernel(const GemmArgs p) {
  constexpr int NC = 8, NP = 4, NT = RING_THREADS;
  static_assert(WM * WN * KG == NC, "eight consumer waves");
  constexpr int BM = WM * MI * 16, BN = WN * NI * 16;
  constexpr bool BLOCK = is_block(KIND);
  constexpr bool HW = KIND == KIND_FP8_BLOCK_POW2;  // the MFMA applies the block scales
  constexpr bool FOLD = BLOCK && !HW;               // they are applied to each MFMA's result
  constexpr int AG = BM / 8, GROUPS = (BM + BN) / 8;       // copies of one KiB (8 rows) per K block: activations, all
  constexpr int COPIES = KG * GROUPS, CPW = (COPIES + NP - 1) / NP;
  constexpr int KB_BYTES = (BM + BN) * 128;
  constexpr int SA_COPIES = (BM + 63) / 64, S_COPIES = BLOCK ? KG * (SA_COPIES + 1) : 0, SPW = (S_COPIES + NP - 1) / NP;
  constexpr int SK_BYTES = (SA_COPIES + 1) * 256;            // scales of one K block: 64 rows per copy, then the weight scales
  constexpr int STAGE_BYTES = KG * KB_BYTES + (BLOCK ? KG * SK_BYTES : 0);
  constexpr int DUMP = NST * STAGE_BYTES;                    // where the copies land that even out the producers' counts
  constexpr int CPS = CPW + SPW;                             // vector-memory operations per producer and stage
  static_assert((NST - 2) * CPS < 64, "vmcnt holds six bits");
  constexpr int IMG_PITCH = BN * 2 + 16;
  constexpr int LDS = DUMP + ((COPIES % NP || S_COPIES % NP) ? 1024 : 0);
  static_assert(LDS <= 160 * 1024 && BM * IMG_PITCH <= DUMP && (KG - 1) * BM * BN * 4 <= DUMP, "LDS");
  __shared__ __attribute__((aligned(1024))) char smem[LDS];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4, l8 = lane >> 3;
  // Block ids are dealt round-robin to the eight XCDs: every XCD gets one contiguous range of tiles, walked in bands of
  // up to eight tile rows, so that a band's row tiles share the weight tile they read at the same time.
  const int tiles_m = GROUPED ? *static_cast<const int*>(p.ws) : p.tiles_m;
  int tm, tn;
  {
    const int tiles = tiles_m * p.tiles_n;
    if (GROUPED && (int)blockIdx.x >= tiles) return;  // the grid covers the largest possible plan
    const int q = tiles >> 3, rem = tiles & 7;
    const int xcd = (int)blockIdx.x & 7, idx = (int)blockIdx.x >> 3;
    const int tile = xcd * q + (xcd < rem ? xcd : rem) + idx;
    const int H = tiles_m <= 8 ? tiles_m : 4;
    const int width = H * p.tiles_n;
    const int group = tile / width, first_m = group * H;
    const int gsz = (tiles_m - first_m) < H ? (tiles_m - first_m) : H;
    const int in_group = tile - group * width;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
  }
  int m0 = tm * BM, m_end = p.M;
  const int n0 = tn * BN;
  const char* weight = p.b;
  const float* weight_scale = p.sb;
  uint32_t weight_tile = (uint32_t)tn;
  if constexpr (GROUPED) {
    const int* entry = static_cast<const int*>(p.ws) + PLAN_HEADER + PLAN_ENTRY * tm;
    const int expert = __builtin_amdgcn_readfirstlane(entry[0]);
    m0 = __builtin_amdgcn_readfirstlane(entry[1]);
    m_end = __builtin_amdgcn_readfirstlane(entry[2]);
    weight += (int64_t)expert * p.b_expert_stride;
    weight_scale += (int64_t)expert * p.sb_expert_stride;
    static_assert(BN == 128, "a tile's number");
    weight_tile = grouped_weight_tile(p, expert, tn);
  }
  const int nkb = (p.K + 127) >> 7, T = (nkb + KG - 1) / KG;
  const int k_tail = p.K & 127;  // bytes of the last K block, 0 = all of it
  const bool sa_packed = HW && p.sa_packed;  // activation scales as words of four K blocks' exponent bytes
  const int sa_kshift = sa_packed ? 2 : 0;

  const int first = __builtin_amdgcn_readfirstlane(GROUPED ? first_k_step(p, weight_tile, T) : first_k_step_shared(p, weight_tile, T));  // stage t holds K step (t + first) % T

  using acc_t = typename std::conditional<float_acc(KIND), v4f, v4i>::type;
  acc_t acc[MI][NI];
  const int kg = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
  const int wrow = wm * MI * 16, wcol = wn * NI * 16;

  if (wave >= NC) {
    // ---- producers: copy c of a stage brings 8 rows of K block c / GROUPS
    const int pw = wave - NC;
    const v4u ra = make_rsrc_sgpr(p.a, p.a_bytes), rb = make_rsrc_sgpr(weight, p.b_bytes);
    const uint32_t chunk_even = (uint32_t)(((lane & 7) ^ l8) & 7) * 16u, chunk_odd = chunk_even ^ 16u;
    const uint32_t lane_a = (uint32_t)(m0 + l8) * p.lda, lane_b = (uint32_t)(n0 + l8) * p.ldb;
    const uint32_t base = lds_addr(smem);
    v4u rsa = ra, rsb = ra;
    uint32_t off_sb = OOB;
    if constexpr (BLOCK) {
      const int nblocks = (p.N + 127) >> 7;
      rsa = make_rsrc_sgpr(p.sa, (uint32_t)(((int64_t)(p.M - 1) * p.sa_stride_m + (int64_t)((nkb - 1) >> sa_kshift) * p.sa_stride_k + 1) * 4));
      rsb = make_rsrc_sgpr(weight_scale, (uint32_t)(((int64_t)(nblocks - 1) * p.sb_stride_n + (int64_t)(nkb - 1) * p.sb_stride_k + 1) * 4));
      const int nb = (n0 >> 7) + lane;
      off_sb = (lane < 3 && nb < nblocks) ? (uint32_t)(nb * p.sb_stride_n * 4) : OOB;
    }
    int t_copy = first;  // the K step that the next copies bring
    auto issue = [&](int slot) __attribute__((always_inline)) {
      const int t = t_copy;
      t_copy = t + 1 == T ? 0 : t + 1;
      const uint32_t st = base + (uint32_t)slot * STAGE_BYTES;
#pragma unroll
      for (int j = 0; j < CPW; ++j) {
        const int c = pw + NP * j;  // (uniform: scalar arithmetic)
        const int q = KG == 1 ? 0 : c / GROUPS, gi = c - q * GROUPS;
        const int u = t * KG + q;
        const bool live = u < nkb && (COPIES % NP == 0 || c < COPIES);
        uint32_t kill = live ? 0u : OOB;
        const uint32_t k0 = live ? (uint32_t)u * 128u : 0u;
        const uint32_t dst = (COPIES % NP == 0 || c < COPIES) ? st + (uint32_t)c * 1024u : base + DUMP;
        const bool is_a = gi < AG;
        const int row8 = is_a ? gi : gi - AG;
        const uint32_t chunk = (row8 & 1) ? chunk_odd : chunk_even;
        if (k_tail && u == nkb - 1 && chunk >= (uint32_t)k_tail) kill = OOB;
        const uint32_t voff = (is_a ? lane_a + (uint32_t)(row8 * 8) * p.lda : lane_b + (uint32_t)(row8 * 8) * p.ldb) + chunk;
        if (is_a) lds_copy16(ra, dst, voff | kill, k0);
        else lds_copy16(rb, dst, voff | kill, k0);
      }
      if constexpr (BLOCK) {
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
          const int c = pw + NP * j;
          const int q = c / (SA_COPIES + 1), r = c - q * (SA_COPIES + 1);
          const int u = t * KG + q;
          const bool slot_ok = S_COPIES % NP == 0 || c < S_COPIES;
          const bool live = u < nkb && slot_ok;
          const uint32_t kill = live ? 0u : OOB;
          const uint32_t kb = live ? (uint32_t)u : 0u;
          const uint32_t dst = slot_ok ? st + KG * KB_BYTES + (uint32_t)c * 256u : base + DUMP;
          if (r < SA_COPIES) {
            const int row = m0 + r * 64 + lane;
            const uint32_t off = row < p.M ? (uint32_t)(row * p.sa_stride_m * 4) : OOB;
            lds_copy4(rsa, dst, off | kill, (kb >> sa_kshift) * (uint32_t)(p.sa_stride_k * 4));
          } else {
            lds_copy4(rsb, dst, off_sb | kill, kb * (uint32_t)(p.sb_stride_k * 4));
          }
        }
      }
    };
#pragma unroll
    for (int t = 0; t < NST - 1; ++t)
      if (t < T) issue(t);
    int slot = NST - 1;
    for (int t = 0; t < T; ++t) {
      const int younger = T - 1 - t < NST - 2 ? T - 1 - t : NST - 2;
      if (younger >= 4) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * CPS < 63 ? 4 * CPS : 63) : "memory");
      else if (younger == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * CPS < 63 ? 3 * CPS : 63) : "memory");
      else if (younger == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * CPS < 63 ? 2 * CPS : 63) : "memory");
      else if (younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CPS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (t + NST - 1 < T) {
        issue(slot);
        slot = slot + 1 == NST ? 0 : slot + 1;
      }
    }
    __builtin_amdgcn_s_barrier();
  } else {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    const int sw = (r16 & 7) ^ (r16 >> 3);
    const int lane_off0 = r16 * 128 + (((2 * g) ^ sw) * 16);
    const int lane_off1 = lane_off0 ^ 16;
    auto read_frag = [&](const char* q) -> v8i {
      v4i lo = *reinterpret_cast<const v4i*>(q + lane_off0);
      v4i hi = *reinterpret_cast<const v4i*>(q + lane_off1);
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    // The operand with fewer fragments is held in registers for a K block, the other one streams through two.
    constexpr bool HOLD_A = MI < NI;
    constexpr int NH = HOLD_A ? MI : NI, NO = HOLD_A ? NI : MI;
    // EARLY: the streamed fragments run two ahead and the barrier stands in front of the last two of them, so that the next stage's
    // first ones are read under twice as many MFMAs.  Block-INT8 2 % (157 shapes, weights in the last-level cache or from HBM alike;
    // 1000 x 5120 x 5120 37.7 -> 36.4 us), scales applied by the MFMA 1.5 % (136 shapes); the other kinds 0.5 % with one shape in twelve
    // 2 % slower, and they stay as they were.  The held fragments doubled as well, so that they too are read ahead: 1 % slower.
    constexpr bool EARLY = NO >= 3 && (KIND == KIND_I8_BLOCK || HW);
    constexpr bool ONE_SB = BN % 128 == 0 && 128 % (NI * 16) == 0;  // a wave's columns lie in one block of weight scales
    constexpr int NSB = ONE_SB ? 1 : NI;
    v8i held[NH], cur, ahead;  // ahead (EARLY): the streamed operand's next fragment
    float sfa[MI], sfb[NSB];
    const int kb_off = KG == 1 ? 0 : kg * KB_BYTES, sc_off = KG * KB_BYTES + (KG == 1 ? 0 : kg * SK_BYTES);
    auto frag_a = [&](const char* st, int i) { return read_frag(st + kb_off + (wrow + i * 16) * 128); };
    auto frag_w = [&](const char* st, int j) { return read_frag(st + kb_off + BM * 128 + (wcol + j * 16) * 128); };
    auto frag_h = [&](const char* st, int h) { return HOLD_A ? frag_a(st, h) : frag_w(st, h); };
    auto frag_o = [&](const char* st, int o) { return HOLD_A ? frag_w(st, o) : frag_a(st, o); };
    auto read_sa = [&](const char* st, int i) { sfa[i] = *reinterpret_cast<const float*>(st + sc_off + (wrow + i * 16 + r16) * 4); };
    auto read_sb = [&](const char* st, int j) {
      const int nb = ONE_SB ? wcol >> 7 : ((n0 & 127) + wcol + j * 16) >> 7;
      sfb[j] = *reinterpret_cast<const float*>(st + sc_off + SA_COPIES * 256 + nb * 4);
    };
    auto step = [&](const char* st, const char* sn, int t, auto read_tag) {
      constexpr int LAST = EARLY ? NO - 2 : NO - 1;  // the next stage is read from this fragment on
      constexpr bool READ = decltype(read_tag)::value;
      v4f part_prev = {0.f, 0.f, 0.f, 0.f};
      float sc_prev = 0.f;
      float sc[MI];
      if constexpr (FOLD && ONE_SB) {
#pragma unroll
        for (int i = 0; i < MI; ++i) sc[i] = sfa[i] * sfb[0];
      }
      int ea[MI], eb[NSB];  // HW: the exponent bytes of the K block's scales
      if constexpr (HW) {
#pragma unroll
        for (int i = 0; i < MI; ++i) ea[i] = ue8m0_at(sfa[i], sa_packed ? 8 * (((t + first < T ? t + first : t + first - T) * KG + kg) & 3) : 23);
#pragma unroll
        for (int j = 0; j < NSB; ++j) eb[j] = ue8m0_of(sfb[j]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        v8i nxt = cur, nxt2 = ahead;
        float so[NH];
        if constexpr (FOLD) {
#pragma unroll
          for (int h = 0; h < NH; ++h) so[h] = ONE_SB ? sc[HOLD_A ? h : o] : (HOLD_A ? sfa[h] * sfb[o] : sfa[o] * sfb[h]);
        }
        if (o == LAST) {
          __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0_only());
          __builtin_amdgcn_s_barrier();  // every wave has read this stage; the next one has landed
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int h = 0; h < NH; ++h) {
          const int i = HOLD_A ? h : o, j = HOLD_A ? o : h;
          const v8i &w = HOLD_A ? cur : held[h], &a = HOLD_A ? held[h] : cur;
          v4f part = {0.f, 0.f, 0.f, 0.f};
          if constexpr (FOLD) {
            part = block_mfma<KIND>(w, a);
          } else if constexpr (HW) {
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, a, acc[i][j], 0, 0, 0, eb[ONE_SB ? 0 : j], 0, ea[i]);
          } else if constexpr (KIND == KIND_FP8_ROWCOL) {
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, a, acc[i][j], 0, 0, 0, 0, 0, 0);
          } else {
            const v4i b0 = {w[0], w[1], w[2], w[3]}, b1 = {w[4], w[5], w[6], w[7]};
            const v4i a0 = {a[0], a[1], a[2], a[3]}, a1 = {a[4], a[5], a[6], a[7]};
            acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b0, a0, acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b1, a1, acc[i][j], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (EARLY) {
            if (h == 0) {
              if (o + 2 < NO) nxt2 = frag_o(st, o + 2);
              else if constexpr (READ) nxt2 = frag_o(sn, o + 2 - NO);
            }
          } else if (o + 1 < NO) {
            if (h == 0) nxt = frag_o(st, o + 1);
          }
          if (READ && o == NO - 1) {
            held[h] = frag_h(sn, h);
            if (!EARLY && h == 0) nxt = frag_o(sn, 0);
            if constexpr (BLOCK) {
#pragma unroll
              for (int q = 0; q < MI; ++q)
                if (q * NH / MI == h) read_sa(sn, q);
#pragma unroll
              for (int q = 0; q < NSB; ++q)
                if (q * NH / NSB == h) read_sb(sn, q);
            }
          }
          if constexpr (FOLD) {
            if (o * NH + h > 0) {
              const int po = (o * NH + h - 1) / NH, ph = (o * NH + h - 1) % NH;
              acc_t& d = acc[HOLD_A ? ph : po][HOLD_A ? po : ph];
#pragma unroll
              for (int e = 0; e < 4; ++e) d[e] = __builtin_fmaf(block_value<KIND>(part_prev[e]), sc_prev, d[e]);
            }
            part_prev = part;
            sc_prev = so[h];
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (EARLY) cur = ahead, ahead = nxt2;
        else cur = nxt;
      }
      if constexpr (FOLD) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[MI - 1][NI - 1][e] = __builtin_fmaf(block_value<KIND>(part_prev[e]), sc_prev, acc[MI - 1][NI - 1][e]);
      }
    };
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int h = 0; h < NH; ++h) held[h] = frag_h(smem, h);
    cur = frag_o(smem, 0);
    if constexpr (EARLY) ahead = frag_o(smem, 1);
    if constexpr (BLOCK) {
#pragma unroll
      for (int i = 0; i < MI; ++i) read_sa(smem, i);
#pragma unroll
      for (int j = 0; j < NSB; ++j) read_sb(smem, j);
    }
    const char* st = smem;
    int slot = 0;
    for (int t = 0; t + 1 < T; ++t) {
      slot = slot + 1 == NST ? 0 : slot + 1;
      const char* sn = smem + slot * STAGE_BYTES;
      step(st, sn, t, std::true_type{});
      st = sn;
    }
    step(st, st, T - 1, std::false_type{});
  }
  // every stage is free from here on
  if constexpr (KG > 1) {
    constexpr int PLANE = BM * BN * 4;
    char* const mine = smem + (wm * WN + wn) * MI * NI * 1024 + lane * 16;
    if (wave < NC && kg > 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) *reinterpret_cast<acc_t*>(mine + (kg - 1) * PLANE + (i * NI + j) * 1024) = acc[i][j];
    }
    __syncthreads();
    if (kg == 0) {
#pragma unroll
      for (int q = 0; q < KG - 1; ++q)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] += *reinterpret_cast<const acc_t*>(mine + q * PLANE + (i * NI + j) * 1024);
    }
    __syncthreads();
  }
  const bool owner = wave < NC && kg == 0;
  if (owner) {
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = wrow + i * 16 + r16, m = m0 + row;
      float sam = 1.f;
      if constexpr (KIND == KIND_FP8_ROWCOL || KIND == KIND_I8_ROWCOL) sam = p.sa[m < p.M ? m : p.M - 1];
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int col = wcol + j * 16 + g * 4, n = n0 + col;
        if (n < p.N) {
          float o[4];
          values4<KIND, OUT_DT>(p, n, acc[i][j], sam, o);
          store4<OUT_DT>(smem + row * IMG_PITCH, col, o[0], o[1], o[2], o[3]);
        }
      }
    }
  }
  __syncthreads();
  constexpr int CH = BN / 8;
  for (int c = threadIdx.x; c < BM * CH; c += NT) {
    const int row = c / CH, cc = c % CH;
    if (m0 + row < m_end && n0 + cc * 8 < p.N)
      *reinterpret_cast<v4i*>(reinterpret_cast<char*>(p.out) + ((int64_t)(m0 + row) * p.ldo + n0 + cc * 8) * 2) =
          *reinterpret_cast<const v4i*>(smem + row * IMG_PITCH + cc * 16);
  }
}

template <int KIND, int OUT_DT>
static void launch_ring_config(GemmArgs& p, int config, hipStream_t st) {
  p.tiles_m = (p.M + RING_BM[config] - 1) / RING_BM[config];
  p.tiles_n = (p.N + RING_BN[config] - 1) / RING_BN[config];
  p.splits = 1;
  const dim3 grid((uint32_t)(p.tiles_m * p.tiles_n)), block(RING_THREADS);
  switch (config) {
#define SGLQ_RING_CASE(i, wm, wn, kg, mi, ni, nst) \
  case i: gemm_ring_kernel<KIND, OUT_DT, wm, wn, kg, mi, ni, nst><<<grid, block, 0, st>>>(p); break;
    SGLQ_RING_CONFIGS(SGLQ_RING_CASE)
#undef SGLQ_RING_CASE
  }
}

// A group of problems: the grid is sized for the largest possible plan, p.tiles_m row tiles.
template <int KIND, int OUT_DT>
static void launch_ring_grouped_config(GemmArgs& p, int config, hipStream_t st) {
  p.tiles_n = (p.N + RING_BN[config] - 1) / RING_BN[config];
  p.splits = 1;
  const dim3 grid((uint32_t)(p.tiles_m * p.tiles_n)), block(RING_THREADS);
  switch (config) {
#define SGLQ_RING_CASE(i, wm, wn, kg, mi, ni, nst)                                                                              \
  case i:                                                                                                                        \
    if constexpr (RING_GROUPED[i]) gemm_ring_kernel<KIND, OUT_DT, wm, wn, kg, mi, ni, nst, true><<<grid, block, 0, st>>>(p);       \
    break;
    SGLQ_RING_CONFIGS(SGLQ_RING_CASE)
#undef SGLQ_RING_CASE
  }
}

template <int KIND>
static void launch_ring_kind(GemmArgs& p, int config, int out_dtype, hipStream_t st) {
  if (out_dtype == SGLQ_BF16) launch_ring_config<KIND, SGLQ_BF16>(p, config, st);
  else if constexpr (KIND != KIND_FP8_BLOCK_POW2) launch_ring_config<KIND, SGLQ_FP16>(p, config, st);
}

}  // namespace sglq
