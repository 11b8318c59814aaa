// gemm_kwave_kernel (see gemm_kwave.h) and its launcher for one kind.
#pragma once
#include "gemm_kwave.h"

namespace sglq {

// The plan of one wave and K block.  A K block is UA units of activation rows (a unit: 32 rows of 128 bytes, 4 KiB, four
// copies; the last one 16 rows where MI is odd), then UB units of weight rows.  Units pass through a ring of NU slots in
// that order; step b (0 .. UB - 1) multiplies weight unit b and refills the slots of the units that refills(b) says, in order.
template <int KIND, int MI, int NI>
struct KwavePlan {
  static constexpr bool BLOCK = is_block(KIND);
  static constexpr int BM = 16 * MI, BN = 16 * NI;
  static constexpr int UA = (MI + 1) / 2, UB = NI / 2, UPB = UA + UB;
  static constexpr int SA_COPIES = (BM + 63) / 64, SCP = BLOCK ? SA_COPIES + 1 : 0;  // copies of a K block's scales
  static constexpr int SC_BYTES = 256 * (SA_COPIES + 1), NSC = BLOCK ? 4 : 0;
  // first unit (index in the K block) that step b refills, and one past its last; last unit that step b reads: the next
  // weight unit, or with the K block's last step the next K block's activations and first weight unit
  static constexpr int refill_from(int b) { return b == 0 ? 0 : b == 1 ? UA - 1 : UA + b - 1; }
  static constexpr int refill_to(int b) { return b == UB - 1 ? UPB : refill_from(b + 1); }
  static constexpr int last_read(int b) { return b == UB - 1 ? UPB + UA : UA + b + 1; }
  // units under way across the wait of every step with a ring of `nu` slots, at least
  static constexpr int under_way(int nu) {
    int least = nu;
    for (int b = 0; b < UB; ++b) least = nu + refill_from(b) - last_read(b) - 1 < least ? nu + refill_from(b) - last_read(b) - 1 : least;
    return least;
  }
  // Slots: the code of a K block is repeated for each of the PER positions that it can have in the ring, so that every
  // slot is a constant; the ring is what fits, shortened by up to two slots where that needs fewer repetitions and two units
  // stay under way across every wait.  Fewer repetitions are worth 2-3 % (block-FP8 on 64 x 64 tiles, eight slots and two of
  // them against nine and nine); a ring that a wait drains costs more (80 x 64 and 96 x 64, seven slots: 9 % slower than nine
  // on average of 34 shapes, 33 % at most; in place 112 x 64 and 128 x 64, one unit left: 1 %).
  static constexpr int gcd(int x, int y) { return y == 0 ? x : gcd(y, x % y); }
  static constexpr int period(int nu) { return nu / gcd(nu, UPB); }
  static constexpr int NU_MAX = (160 * 1024 / 4 - NSC * SC_BYTES) / 4096;
  static constexpr int shorter(int x, int y) { return under_way(y) >= 2 && period(y) < period(x) ? y : x; }
  static constexpr int NU = shorter(shorter(NU_MAX, NU_MAX - 1), NU_MAX - 2), PER = period(NU);
  static_assert(NU >= UPB && under_way(NU) >= 2, "a wait does not drain the ring");
  static constexpr int WAVE_BYTES = NU * 4096 + NSC * SC_BYTES;
  static_assert(UB >= 2 && NI % 4 == 0 && (NU + UPB - 1) / UPB <= 4, "an even number of steps, the waves' shares of the columns, slots of scales");
  // copies of unit u, counted on over the K blocks (a K block's scales go in front of its first unit)
  static constexpr int copies(int u) { return (u % UPB == UA - 1 && (MI & 1) ? 2 : 4) + (u % UPB == 0 ? SCP : 0); }
  // copies under way when step b starts that are younger than the last unit it reads
  static constexpr int younger(int b) {
    int n = 0;
    for (int u = last_read(b) + 1; u < NU + refill_from(b); ++u) n += copies(u);
    return n;
  }
  // refill copies of step b in the order in which they are issued: number, and for copy c its unit and its index there
  // (below SCP of a K block's first unit: scales)
  static constexpr int refills(int b) {
    int n = 0;
    for (int u = refill_from(b); u < refill_to(b); ++u) n += copies(u + NU);
    return n;
  }
  static constexpr int refill_unit(int b, int c) {
    int u = refill_from(b);
    while (c >= copies(u + NU)) c -= copies(u++ + NU);
    return u;
  }
  static constexpr int refill_index(int b, int c) {
    for (int u = refill_from(b); c >= copies(u + NU); ++u) c -= copies(u + NU);
    return c;
  }
  // ... how many of them have been issued behind MFMA m (0 .. 2 MI - 1) of step b.  In step 0 a slot of activations is free
  // behind the first MFMA that uses its last fragment; in the other steps all of their slots are free, the last step's
  // last one behind its second MFMA.
  static constexpr int refilled(int b, int m) {
    const int n = refills(b), steps = 2 * MI;
    if (m < 0) return 0;
    if (b > 0) return (m + 1) * n / steps;
    int free = 0;
    for (int u = refill_from(b); u < refill_to(b); ++u)
      if (4 * u + 3 <= m) free += copies(u + NU);
    return free;
  }
  static constexpr int younger_start() {
    int n = 0;
    for (int u = UA + 1; u < NU; ++u) n += copies(u);
    return n;
  }
};

// lds_copy16 to `base` and a constant
template <int DST>
SGLQ_DEV void lds_copy16_at(v4u rsrc, uint32_t base, uint32_t voff, uint32_t soff) {
  asm volatile("s_add_u32 m0, %0, %4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" : : "s"(base), "v"(voff), "s"(rsrc), "s"(soff), "n"(DST) : "memory", "scc");
}

template <int KIND, int OUT_DT, int MI, int NI>
SGLQ_DEV void kwave_body(const GemmArgs& p) {
  using Plan = KwavePlan<KIND, MI, NI>;
  constexpr int BM = Plan::BM, BN = Plan::BN, UA = Plan::UA, UB = Plan::UB, UPB = Plan::UPB, NU = Plan::NU;
  constexpr bool BLOCK = is_block(KIND);
  constexpr bool FOLD = BLOCK;  // the block scales are applied to each MFMA's result
  static_assert(KIND != KIND_FP8_BLOCK_POW2 && KIND != KIND_I8_RAW, "not built");
  constexpr int NW = 4;
  constexpr int IMG_PITCH = BN * 2 + 16;
  constexpr int LDS = 160 * 1024;  // the rings; then partial sums and the output's image
  static_assert(NW * Plan::WAVE_BYTES <= LDS && BM * IMG_PITCH <= LDS, "LDS");
  static_assert(!BLOCK || BN == 64 || BN == 128, "a tile's columns lie in one block of weight scales");
  __shared__ __attribute__((aligned(1024))) char smem[LDS];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4, l8 = lane >> 3;
  // (tiles over the XCDs as in gemm_ring_kernel: bands of up to eight tile rows, whose row tiles share the weight tile)
  int tm, tn;
  {
    const int tiles = p.tiles_m * p.tiles_n;
    const int q = tiles >> 3, rem = tiles & 7;
    const int xcd = (int)blockIdx.x & 7, idx = (int)blockIdx.x >> 3;
    const int tile = xcd * q + (xcd < rem ? xcd : rem) + idx;
    const int H = p.tiles_m <= 8 ? p.tiles_m : 4;
    const int width = H * p.tiles_n;
    const int group = tile / width, first_m = group * H;
    const int gsz = (p.tiles_m - first_m) < H ? (p.tiles_m - first_m) : H;
    const int in_group = tile - group * width;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
  }
  const int m0 = tm * BM, n0 = tn * BN;
  const int nkb = p.K >> 7;
  const int T = (nkb - wave + NW - 1) / NW;  // this wave's K blocks: wave, wave + 4, ...

  using acc_t = typename std::conditional<float_acc(KIND), v4f, v4i>::type;
  acc_t acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = acc_t{0, 0, 0, 0};

  if (T > 0) {
    // ---- copies: copy j of a unit brings its rows 8 j .. + 7, lane l chunk (l % 8) ^ swz of row l / 8
    const v4u ra = make_rsrc_sgpr(p.a, p.a_bytes), rb = make_rsrc_sgpr(p.b, p.b_bytes);
    const uint32_t ring = lds_addr(smem) + (uint32_t)(wave * Plan::WAVE_BYTES);
    uint32_t voff_a[4], voff_b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t chunk = (uint32_t)((((lane & 7) ^ l8) & 7) * 16) ^ (j & 1 ? 16u : 0u);
      voff_a[j] = (uint32_t)(m0 + l8 + 8 * j) * p.lda + chunk;
      voff_b[j] = (uint32_t)(n0 + l8 + 8 * j) * p.ldb + chunk;
    }
    v4u rsa = ra, rsb = ra;
    uint32_t voff_sa[Plan::SA_COPIES], voff_sb = OOB;
    if constexpr (BLOCK) {
      const int nblocks = (p.N + 127) >> 7;
      rsa = make_rsrc_sgpr(p.sa, (uint32_t)(((int64_t)(p.M - 1) * p.sa_stride_m + (int64_t)(nkb - 1) * p.sa_stride_k + 1) * 4));
      rsb = make_rsrc_sgpr(p.sb, (uint32_t)(((int64_t)(nblocks - 1) * p.sb_stride_n + (int64_t)(nkb - 1) * p.sb_stride_k + 1) * 4));
      if (lane == 0) voff_sb = (uint32_t)((n0 >> 7) * p.sb_stride_n * 4);
#pragma unroll
      for (int c = 0; c < Plan::SA_COPIES; ++c) {
        const int row = m0 + c * 64 + lane;
        voff_sa[c] = row < p.M ? (uint32_t)(row * p.sa_stride_m * 4) : OOB;
      }
    }
    // copy j of unit u (both static) of wave K block t into slot `slot`; a K block past the last one is zero fill
    const int first = __builtin_amdgcn_readfirstlane(first_k_step_shared(p, (uint32_t)tn, T));
    const int behind = first * NW + wave, past = behind + NW * T;  // (the t-th K block, once past the last one it is `T` back)
    auto k_block_at = [&](int t) __attribute__((always_inline)) {
      const int kb = behind + NW * t;
      return kb < nkb ? kb : kb < past ? kb - NW * T : nkb;
    };
    auto k_offset = [&](int t) __attribute__((always_inline)) -> uint32_t {
      const int kb = k_block_at(t);
      return kb < nkb ? (uint32_t)kb * 128u : OOB;
    };
    auto copy_unit = [&](auto u_tag, auto j_tag, auto slot_tag, uint32_t k0) __attribute__((always_inline)) {
      constexpr int u = decltype(u_tag)::value, j = decltype(j_tag)::value, dst = decltype(slot_tag)::value * 4096 + j * 1024;
      const uint32_t soff = u < UA ? k0 + (uint32_t)(u * 32) * p.lda : k0 + (uint32_t)((u - UA) * 32) * p.ldb;
      lds_copy16_at<dst>(u < UA ? ra : rb, ring, u < UA ? voff_a[j] : voff_b[j], soff);
    };
    auto copy_scales = [&](int c, int t) __attribute__((always_inline)) {
      if constexpr (BLOCK) {
        const int kb = k_block_at(t);
        const uint32_t dst = ring + NU * 4096 + (uint32_t)(t & (Plan::NSC - 1)) * Plan::SC_BYTES + (uint32_t)c * 256u;
        if (c < Plan::SA_COPIES) lds_copy4(rsa, dst, voff_sa[c], kb < nkb ? (uint32_t)(kb * p.sa_stride_k * 4) : SC_NONE);
        else lds_copy4(rsb, dst, voff_sb, kb < nkb ? (uint32_t)(kb * p.sb_stride_k * 4) : SC_NONE);
      }
    };
    // ---- operands
    const int sw = (r16 & 7) ^ (r16 >> 3);
    const char* const rd0 = smem + wave * Plan::WAVE_BYTES + r16 * 128 + (((2 * g) ^ sw) * 16);
    const char* const rd1 = smem + wave * Plan::WAVE_BYTES + r16 * 128 + (((2 * g + 1) ^ sw) * 16);
    auto read_frag = [&](int slot, int f) __attribute__((always_inline)) -> v8i {
      const v4i lo = *reinterpret_cast<const v4i*>(rd0 + slot * 4096 + f * 2048);
      const v4i hi = *reinterpret_cast<const v4i*>(rd1 + slot * 4096 + f * 2048);
      return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    v8i a[MI], w[2][2];  // w[b & 1]: weight unit b
    float sfa[MI], sfb;
    const char* const sc_rd = smem + wave * Plan::WAVE_BYTES + NU * 4096;
    auto read_scales = [&](int t) __attribute__((always_inline)) {
      if constexpr (BLOCK) {
        const char* s = sc_rd + (t & (Plan::NSC - 1)) * Plan::SC_BYTES;
#pragma unroll
        for (int i = 0; i < MI; ++i) sfa[i] = *reinterpret_cast<const float*>(s + (i * 16 + r16) * 4);
        sfb = *reinterpret_cast<const float*>(s + Plan::SA_COPIES * 256);
      }
    };

    // ---- start: the ring filled, the first K block's activations, first weight unit and scales read
    static_for<NU>([&](auto u_tag) __attribute__((always_inline)) {
      constexpr int u = decltype(u_tag)::value, scales = u % UPB == 0 ? Plan::SCP : 0;
#pragma unroll
      for (int c = 0; c < scales; ++c) copy_scales(c, u / UPB);
      static_for<Plan::copies(u) - scales>([&](auto j_tag) __attribute__((always_inline)) {
        copy_unit(std::integral_constant<int, u % UPB>{}, j_tag, u_tag, k_offset(u / UPB));
      });
    });
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Plan::younger_start()) : "memory");
#pragma unroll
    for (int i = 0; i < MI; ++i) a[i] = read_frag(i / 2, i & 1);
#pragma unroll
    for (int f = 0; f < 2; ++f) w[0][f] = read_frag(UA, f);
    read_scales(0);

    // one K block, the ring's slot of its first unit is x UPB % NU
    auto k_block = [&](auto x_tag, int t) __attribute__((always_inline)) {
      constexpr int x = decltype(x_tag)::value;
      float sc[MI];
      constexpr int LAG = 2;  // MFMAs between a product and its folding
      v4f part[LAG + 1];
      const uint32_t k_refill[3] = {k_offset(t + NU / UPB), k_offset(t + NU / UPB + 1), k_offset(t + NU / UPB + 2)};
      static_for<UB>([&](auto b_tag) __attribute__((always_inline)) {
        constexpr int b = decltype(b_tag)::value;
        constexpr bool last = b == UB - 1;
        // the next unit has landed (with the last step: the next K block's activations too); this wave alone uses the ring
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Plan::younger(b)) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        constexpr int next = (x * UPB + (last ? UPB + UA : UA + b + 1)) % NU;
        w[(b + 1) & 1][0] = read_frag(next, 0);
        w[(b + 1) & 1][1] = read_frag(next, 1);
        // MFMA q of a step is of fragments (q / 2, 2 b + q % 2)
        auto fold = [&](int q, int fb) __attribute__((always_inline)) {
          acc_t& d = acc[q / 2][2 * fb + (q & 1)];
#pragma unroll
          for (int e = 0; e < 4; ++e) d[e] = __builtin_fmaf(block_value<KIND>(part[(2 * MI * fb + q) % (LAG + 1)][e]), sc[q / 2], d[e]);
        };
        if constexpr (FOLD && b == 0) {
#pragma unroll
          for (int i = 0; i < MI; ++i) sc[i] = sfa[i] * sfb;
        }
        __builtin_amdgcn_sched_barrier(0);
        static_for<2 * MI>([&](auto q_tag) __attribute__((always_inline)) {
          constexpr int q = decltype(q_tag)::value, i = q / 2, j = 2 * b + (q & 1);
          const v8i &wf = w[b & 1][q & 1], &af = a[i];
          if constexpr (FOLD) {
            part[(2 * MI * b + q) % (LAG + 1)] = block_mfma<KIND>(wf, af);
          } else if constexpr (KIND == KIND_FP8_ROWCOL) {
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, af, acc[i][j], 0, 0, 0, 0, 0, 0);
          } else {
            const v4i b0 = {wf[0], wf[1], wf[2], wf[3]}, b1 = {wf[4], wf[5], wf[6], wf[7]};
            const v4i a0 = {af[0], af[1], af[2], af[3]}, a1 = {af[4], af[5], af[6], af[7]};
            acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b1, a1, __builtin_amdgcn_mfma_i32_16x16x64_i8(b0, a0, acc[i][j], 0, 0, 0), 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (last && (q & 1)) {  // this activation fragment has had its last use
            a[i] = read_frag((x * UPB + UPB + i / 2) % NU, i & 1);
          }
          constexpr int c0 = Plan::refilled(b, q - 1), c1 = Plan::refilled(b, q);
          static_for<c1 - c0>([&](auto c_tag) __attribute__((always_inline)) {
            constexpr int c = c0 + decltype(c_tag)::value;
            constexpr int u = Plan::refill_unit(b, c) + NU, n = Plan::refill_index(b, c), scales = u % UPB == 0 ? Plan::SCP : 0;
            if constexpr (n < scales) copy_scales(n, t + u / UPB);
            else
              copy_unit(std::integral_constant<int, u % UPB>{}, std::integral_constant<int, n - scales>{},
                        std::integral_constant<int, (x * UPB + u) % NU>{}, k_refill[u / UPB - NU / UPB]);
          });
          if constexpr (FOLD) {
            if constexpr (q >= LAG) fold(q - LAG, b);
            else if constexpr (b > 0) fold(2 * MI + q - LAG, b - 1);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (last) {
          read_scales(t + 1);
          if constexpr (FOLD) {
#pragma unroll
            for (int q = 2 * MI - LAG; q < 2 * MI; ++q) fold(q, b);
          }
        }
      });
    };
    int t = 0;
    while (true) {
      bool more = true;
      static_for<Plan::PER>([&](auto x_tag) __attribute__((always_inline)) {
        if (more) {
          k_block(x_tag, t);
          more = ++t < T;
        }
      });
      if (!more) break;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (what the last refills, zero fill, still write into LDS)
  }

  // ---- the waves' sums, added in the order of the waves: fragment f by wave f % 4.  PR fragment rows at a time.
  constexpr int PR = MI * NI <= 40 ? MI : MI / 2, NQ = PR * NI / NW;
  static_assert(NW * PR * NI * 1024 <= 160 * 1024 && MI % PR == 0, "all partial sums of a pass in LDS");
  constexpr bool ROWCOL = !is_block(KIND);
  char* const mine = smem + lane * 16;
  v4f img[MI / PR][NQ];  // (16-bit values, four per fragment and lane, wait here for the image: LDS is still being read)
#pragma unroll
  for (int ps = 0; ps < MI / PR; ++ps) {
    float sam[NQ];
    v4f sbn[NQ];
    float bias[NQ][4];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int f = wave + NW * q, m = m0 + (ps * PR + f / NI) * 16 + r16, n = n0 + f % NI * 16 + 4 * g;
      if constexpr (ROWCOL) {
        sam[q] = p.sa[m < p.M ? m : p.M - 1];
        sbn[q] = *reinterpret_cast<const v4f*>(p.sb + (n < p.N ? n : p.N - 4));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[q][e] = 0.f;
      if (p.bias) load_bias4<OUT_DT>(p.bias, n < p.N ? n : p.N - 4, bias[q]);
    }
    __syncthreads();  // (every wave is done with the ring, or with reading the pass before)
#pragma unroll
    for (int i = 0; i < PR; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) *reinterpret_cast<acc_t*>(mine + ((wave * PR + i) * NI + j) * 1024) = acc[ps * PR + i][j];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      acc_t s = *reinterpret_cast<const acc_t*>(mine + (wave + NW * q) * 1024);
#pragma unroll
      for (int x = 1; x < NW; ++x) s += *reinterpret_cast<const acc_t*>(mine + (x * PR * NI + wave + NW * q) * 1024);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float o;
        if constexpr (is_block(KIND)) o = p.bias ? round_out<OUT_DT>(s[e]) + bias[q][e] : s[e];
        else if constexpr (KIND == KIND_I8_ROWCOL) o = __builtin_fmaf((float)s[e], sbn[q][e] * sam[q], bias[q][e]);
        else o = __builtin_fmaf(sam[q], sbn[q][e] * s[e], bias[q][e]);
        img[ps][q][e] = o;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int ps = 0; ps < MI / PR; ++ps)
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int f = wave + NW * q;
      store4<OUT_DT>(smem + ((ps * PR + f / NI) * 16 + r16) * IMG_PITCH, f % NI * 16 + 4 * g, img[ps][q][0], img[ps][q][1], img[ps][q][2], img[ps][q][3]);
    }
  __syncthreads();
  constexpr int CH = BN / 8;
  for (int c = threadIdx.x; c < BM * CH; c += NW * 64) {
    const int row = c / CH, cc = c % CH;
    if (m0 + row < p.M && n0 + cc * 8 < p.N)
      *reinterpret_cast<v4i*>(reinterpret_cast<char*>(p.out) + ((int64_t)(m0 + row) * p.ldo + n0 + cc * 8) * 2) =
          *reinterpret_cast<const v4i*>(smem + row * IMG_PITCH + cc * 16);
  }
}

template <int KIND, int OUT_DT, int MI, int NI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void gemm_kwave_kernel(const GemmArgs p) {
  kwave_body<KIND, OUT_DT, MI, NI>(p);
}
// The kinds that fold: bounds of 512 lanes (256 are launched) limit the registers to the half that vector instructions reach.
// Given all of them, the compiler puts the products into the other half and copies every one back (four more instructions
// per MFMA: 333 x 4096 x 7168 on 64 x 128 tiles 25.3 us against 23.8).
template <int KIND, int OUT_DT, int MI, int NI>
__global__ __launch_bounds__(512) void gemm_kwave_fold_kernel(const GemmArgs p) {
  kwave_body<KIND, OUT_DT, MI, NI>(p);
}

template <int KIND, int OUT_DT>
static void launch_kwave_config(GemmArgs& p, int config, hipStream_t st) {
  p.tiles_m = (p.M + KWAVE_BM[config] - 1) / KWAVE_BM[config];
  p.tiles_n = (p.N + KWAVE_BN[config] - 1) / KWAVE_BN[config];
  p.splits = 1;
  const dim3 grid((uint32_t)(p.tiles_m * p.tiles_n)), block(256);
  switch (config) {
#define SGLQ_KWAVE_CASE(i, mi, ni) \
  case i:                          \
    if constexpr (!kwave_built(KIND, i)) {} \
    else if constexpr (KIND == KIND_FP8_BLOCK || KIND == KIND_I8_BLOCK) gemm_kwave_fold_kernel<KIND, OUT_DT, mi, ni><<<grid, block, 0, st>>>(p); \
    else gemm_kwave_kernel<KIND, OUT_DT, mi, ni><<<grid, block, 0, st>>>(p); \
    break;
    SGLQ_KWAVE_CONFIGS(SGLQ_KWAVE_CASE)
#undef SGLQ_KWAVE_CASE
  }
}

template <int KIND>
static void launch_kwave_kind(GemmArgs& p, int config, int out_dtype, hipStream_t st) {
  if (out_dtype == SGLQ_BF16) launch_kwave_config<KIND, SGLQ_BF16>(p, config, st);
  else launch_kwave_config<KIND, SGLQ_FP16>(p, config, st);
}

}  // namespace sglq
