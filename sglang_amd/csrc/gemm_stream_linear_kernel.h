// gemm_stream_quant_kernel and gemm_stream_tokenquant_kernel (see gemm_stream_linear.h) and their launcher for one kind.
#pragma once
#include "gemm_stream_linear.h"
#include "quant_device.h"

namespace sglq {

// (arrives in `dst` unseen by the compiler's wait counts, see wait_x.  To the compiler `dst` is written here: a copy or a spill of it in front of
// wait_x would take what was there before.  None of the instantiations has one, and nothing but a look at the code built shows it:
// tests/test_waits_in_code.py follows every way through each, for another compiler, another register budget, another order of these loads.)
SGLQ_DEV void load16(v4u& dst, v4u rsrc, uint32_t voff) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2, 0 offen" : "=v"(dst) : "v"(voff), "s"(rsrc) : "memory");
}
template <int KIND, int NIB, int OUT_DT, int IN_DT, int ROWS>
SGLQ_DEV void stream_linear_body(const GemmArgs& p) {
  static_assert(KIND == KIND_FP8_BLOCK || KIND == KIND_FP8_ROWCOL || KIND == KIND_I8_ROWCOL, "FP8 in groups of 128, FP8 and INT8 per token");
  static_assert(ROWS == 1 || ROWS == 2 || ROWS == 4 || ROWS == 8, "rows of activations");
  constexpr bool BLOCK = KIND == KIND_FP8_BLOCK, IS_FP8 = KIND != KIND_I8_ROWCOL;
  constexpr int BN = NIB * 16, WC = BN / 8, W_BYTES = BN * 128;
  constexpr int NSTAGE = SGLQ_STREAM_NSTAGE, RING_BYTES = NSTAGE * W_BYTES;
  // A K block of a row lies on LPK lanes (a group's scale is formed by each of them: on 16 lanes twice as often as on 8, which take
  // two registers).  A unit is what the wave holds so: SPU steps of ROWS rows in REGS registers; UNITS units, PASS steps, are in registers at a time.
  constexpr int LPK = ROWS == 8 ? 8 : 16, REGS = 16 / LPK, PAIRS = 64 / LPK, SPU = PAIRS / ROWS, UNITS = 16 / REGS, PASS = SPU * UNITS;
  constexpr int UNIT_BYTES = SPU * ROWS * 128;
  static_assert(PASS <= 64, "a step's weight scale on a lane each");
  constexpr int CODES = 4 * RING_BYTES, SCALES = CODES + 4 * 2 * UNIT_BYTES, SFB = SCALES + 4 * 2 * SPU * ROWS * 4;
  static_assert(NIB * 1024 <= RING_BYTES && (NSTAGE - 1) * WC <= 63, "LDS and vmcnt");
  // (one LDS object: rings; the waves' codes of two units; their scales, or the waves' row maxima; the weight scales)
  __shared__ __attribute__((aligned(1024))) char smem[SFB + (BLOCK ? 1024 : 0)];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4, l8 = lane >> 3;
  const int n0 = blockIdx.x * BN;
  const int nkb = p.K >> 7;
  const int nsteps = (nkb - wave + 3) >> 2;  // K blocks wave, wave + 4, ... in turn, from the first_k_step-th on
  const int first = first_k_step(p, (uint32_t)n0 / BN, nsteps);

  const v4u rx = make_rsrc_sgpr(p.a, p.a_bytes), rb = make_rsrc_sgpr(p.b, p.b_bytes);
  // ---- activations into registers, written as assembly like the copies behind them: the compiler would wait for those too
  const int pair = lane / LPK, piece = lane % LPK, q_row = pair % ROWS, q_step = pair / ROWS;  // this lane's row, and its step in a unit
  v4u x[UNITS][REGS];
  // f(u) for the units from step t0 on that there are (in fours: a branch that is not taken for each unit of 16 costs short rows 0.4 us)
  auto for_units = [&](int t0, auto&& f) __attribute__((always_inline)) {
    static_for<UNITS / 4>([&](auto c_tag) __attribute__((always_inline)) {
      constexpr int c = decltype(c_tag)::value;
      if (t0 + 4 * SPU * c < nsteps)
        static_for<4>([&](auto k_tag) __attribute__((always_inline)) {
          constexpr int u = 4 * c + decltype(k_tag)::value;
          if (t0 + SPU * u < nsteps) f(std::integral_constant<int, u>{});
        });
    });
  };
  [[maybe_unused]] v4u rsb = rb;
  [[maybe_unused]] int nb = 0;
  if constexpr (BLOCK) {
    const int nblocks = (p.N + 127) >> 7;
    nb = (n0 >> 7) < nblocks ? n0 >> 7 : nblocks - 1;  // BN divides 128: one block of weight scales
    rsb = make_rsrc_sgpr(p.sb, (uint32_t)(((int64_t)(nblocks - 1) * p.sb_stride_n + (int64_t)(nkb - 1) * p.sb_stride_k + 1) * 4));
  }
  auto step_at = [&](int t) __attribute__((always_inline)) { return first + t < nsteps ? first + t : first + t - nsteps; };
  auto load_x = [&](int t0) __attribute__((always_inline)) {  // of steps t0 .. t0 + PASS - 1, and the weight scales of their K blocks
    for_units(t0, [&](auto u_tag) __attribute__((always_inline)) {
      constexpr int u = decltype(u_tag)::value;
      const int t = t0 + SPU * u + q_step;
      const uint32_t off = (uint32_t)q_row * p.lda + (uint32_t)(wave + 4 * step_at(t)) * 256u + (uint32_t)piece * (16u * REGS);
      const uint32_t voff = t < nsteps && q_row < p.M ? off : OOB;
#pragma unroll
      for (int j = 0; j < REGS; ++j) load16(x[u][j], rx, voff + 16u * j);
    });
    if constexpr (BLOCK) {
      const int t = t0 + lane;
      const bool live = lane < PASS && t < nsteps;
      lds_copy4(rsb, lds_addr(smem) + SFB + wave * 256, live ? (uint32_t)(((wave + 4 * step_at(t)) * p.sb_stride_k + nb * p.sb_stride_n) * 4) : OOB, 0u);
    }
  };
  auto wait_x = [&](auto younger_tag) __attribute__((always_inline)) {  // ... have arrived, `younger` operations behind them may be under way
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(younger_tag)::value) : "memory");
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
#pragma unroll
      for (int j = 0; j < REGS; ++j) asm volatile("" : "+v"(x[u][j]));
    __builtin_amdgcn_sched_barrier(0);
  };
  auto amax16 = [&](const v4u& v, v2us m) __attribute__((always_inline)) {  // sign-stripped bits of the 16-bit type, as integers
#pragma unroll
    for (int w = 0; w < 4; ++w) m = __builtin_elementwise_max(m, __builtin_bit_cast(v2us, v[w] & 0x7fff7fffu));
    return m;
  };
  auto amax_of_block = [&](v2us m) __attribute__((always_inline)) { return group_umax<LPK>(m.x > m.y ? (uint32_t)m.x : (uint32_t)m.y); };
  v2us m16 = {0, 0};
  auto rows_amax = [&](int t0) __attribute__((always_inline)) {
    for_units(t0, [&](auto u_tag) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < REGS; ++j) m16 = amax16(x[decltype(u_tag)::value][j], m16);
    });
  };
  if constexpr (!BLOCK) {  // (longer rows than the registers hold are read twice)
    for (int t0 = PASS; t0 < nsteps; t0 += PASS) {
      load_x(t0);
      wait_x(std::integral_constant<int, 0>{});
      rows_amax(t0);
    }
  }
  load_x(0);

  // ---- the ring: weights only
  const int c16_even = (((lane & 7) ^ l8) & 7) * 16, c16_odd = (((lane & 7) ^ l8 ^ 1) & 7) * 16;
  const uint32_t offw_even = (uint32_t)(n0 + l8) * p.ldb + c16_even, offw_odd = (uint32_t)(n0 + l8) * p.ldb + c16_odd;
  const uint32_t step_w = 8u * p.ldb;
  const uint32_t ring = lds_addr(smem) + (uint32_t)wave * RING_BYTES;
  uint32_t kb = (uint32_t)(wave + 4 * first);  // this wave's next K block to copy
  auto issue_group = [&](int t) __attribute__((always_inline)) {  // all copies of this wave's t-th K block into slot t % NSTAGE
    const uint32_t st = ring + (uint32_t)(t % NSTAGE) * W_BYTES;
    const uint32_t kill = t < nsteps ? 0u : OOB;  // past the end: out of range, the K offset is not bounds-checked
    const uint32_t k0 = t < nsteps ? kb * 128u : 0u;
#pragma unroll
    for (int j = 0; j < WC; ++j)
      lds_copy16(rb, st + j * 1024, (((j & 1) ? offw_odd : offw_even) + j * step_w) | kill, k0);
    kb += 4;
    if (kb >= (uint32_t)nkb) kb = wave;
  };
#pragma unroll
  for (int t = 0; t < NSTAGE - 1; ++t) issue_group(t);

  // ---- the activations are older than every copy of weights: this waits for none of those
  wait_x(std::integral_constant<int, (NSTAGE - 1) * WC>{});
  const int t_row = lane & (ROWS - 1);  // (fragment rows past the last activation row repeat the others; their results are not stored)
  float out_scale = 1.f, q_mul = 1.f;
  float* const sc_lds = reinterpret_cast<float*>(smem + SCALES);
  uint32_t* const red = reinterpret_cast<uint32_t*>(sc_lds);  // [wave][pair]
  if constexpr (!BLOCK) {
    rows_amax(0);
    const uint32_t m = amax_of_block(m16);
    if (piece == 0) red[wave * PAIRS + pair] = m;
  }
  if constexpr (!BLOCK) {
    __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0_only());
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // every lane forms row t_row's scale and multiplier, with the expressions of token_quant_kernel, and fetches its own row's
    uint32_t m = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int q = 0; q < SPU; ++q) m = umax(m, red[w * PAIRS + q * ROWS + t_row]);
    const float amax_x = to_f32_16<IN_DT>((uint16_t)m);
    float mul;
    if constexpr (IS_FP8) {
      out_scale = amax_x / 448.0f;
      mul = (out_scale == 0.f) ? 0.f : 1.0f / out_scale;
    } else {
      const float amax = u2f(umax(f2u(amax_x), f2u(1e-10f)));
      out_scale = amax / 127.0f;
      mul = 127.0f / amax;
    }
    q_mul = u2f((uint32_t)__builtin_amdgcn_ds_bpermute(q_row * 4, (int)f2u(mul)));
  }

  char* const my_codes = smem + CODES + wave * 2 * UNIT_BYTES;
  float* const my_scales = sc_lds + wave * 2 * SPU * ROWS;
  // a unit's codes, in the operand layout: K block by K block, rows of 128 bytes, chunks of 16 swizzled by the row.  A wave's LDS operations
  // execute in order: what it overwrites here it has read before.
  auto quantize = [&](auto u_tag) __attribute__((always_inline)) {
    constexpr int u = decltype(u_tag)::value, buf = u & 1;
    float y_s = 0.f, inv = 0.f;
    if constexpr (BLOCK) {
      v2us m = {0, 0};
#pragma unroll
      for (int j = 0; j < REGS; ++j) m = amax16(x[u][j], m);
      const float amax = u2f(umax(f2u(to_f32_16<IN_DT>((uint16_t)amax_of_block(m))), f2u(p.quant_eps)));
      y_s = div_by(amax, 448.0f, 1.0f / 448.0f);
      inv = 1.0f / y_s;
      if (piece == 0) my_scales[(buf * SPU + q_step) * ROWS + q_row] = y_s;
    }
    v2u codes[REGS];
#pragma unroll
    for (int j = 0; j < REGS; ++j) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xe = to_f32_16<IN_DT>((uint16_t)(x[u][j][e >> 1] >> (16 * (e & 1))));
        if constexpr (BLOCK) v[e] = quantize_elem<false>(xe, y_s, inv, -448.0f, 448.0f);
        else if constexpr (IS_FP8) v[e] = clampf(xe * q_mul, -448.0f, 448.0f);
        else v[e] = clampf(__builtin_roundf(xe * q_mul), -128.0f, 127.0f);
      }
      if constexpr (IS_FP8) codes[j] = Fp8Pack::pack(v);
      else codes[j] = I8Pack::pack(v);
    }
    char* const to = my_codes + buf * UNIT_BYTES + (q_step * ROWS + q_row) * 128;
    if constexpr (REGS == 2) *reinterpret_cast<v4u*>(to + ((piece ^ q_row) & 7) * 16) = v4u{codes[0].x, codes[0].y, codes[1].x, codes[1].y};
    else *reinterpret_cast<v2u*>(to + (((piece >> 1) ^ q_row) & 7) * 16 + (piece & 1) * 8) = codes[0];
  };

  // ---- K loop
  const int sw = (r16 & 7) ^ (r16 >> 3);
  const int lane_off0 = r16 * 128 + (((2 * g) ^ sw) * 16);
  const int lane_off1 = lane_off0 ^ 16;
  auto read_frag = [&](const char* q) __attribute__((always_inline)) -> v8i {
    v4i lo = *reinterpret_cast<const v4i*>(q + lane_off0);
    v4i hi = *reinterpret_cast<const v4i*>(q + lane_off1);
    return v8i{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  const int code_off0 = t_row * 128 + (((2 * g) ^ t_row) & 7) * 16, code_off1 = code_off0 ^ 16;
  const float* const sfb_lds = reinterpret_cast<const float*>(smem + SFB + wave * 256);
  using acc_t = typename std::conditional<IS_FP8, v4f, v4i>::type;
  acc_t acc[NIB];
#pragma unroll
  for (int j = 0; j < NIB; ++j) acc[j] = acc_t{0, 0, 0, 0};
  char* const my_ring = smem + wave * RING_BYTES;
  // step t (of the pass from t0 on), whose K block is number `slot` of the two units in LDS; `ahead` quantizes the next unit while the copies arrive
  auto step = [&](int t, [[maybe_unused]] int t0, int slot, auto&& ahead) __attribute__((always_inline)) {
    issue_group(t + NSTAGE - 1);
    ahead();
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"((NSTAGE - 1) * WC) : "memory");
    const char* st = my_ring + (t % NSTAGE) * W_BYTES;
    v8i wf[NIB];
#pragma unroll
    for (int j = 0; j < NIB; ++j) wf[j] = read_frag(st + j * 16 * 128);
    const char* ct = my_codes + slot * (ROWS * 128);
    const v4i alo = *reinterpret_cast<const v4i*>(ct + code_off0), ahi = *reinterpret_cast<const v4i*>(ct + code_off1);
    const v8i af = v8i{alo[0], alo[1], alo[2], alo[3], ahi[0], ahi[1], ahi[2], ahi[3]};
    float sc = 0.f;
    if constexpr (BLOCK) sc = my_scales[slot * ROWS + t_row] * sfb_lds[t - t0];
#pragma unroll
    for (int j = 0; j < NIB; ++j) {
      if constexpr (BLOCK) {
        const v4f part = block_mfma<KIND>(wf[j], af);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = __builtin_fmaf(part[e], sc, acc[j][e]);
      } else if constexpr (IS_FP8) {
        acc[j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[j], af, acc[j], 0, 0, 0, 0, 0, 0);
      } else {
        const v4i b0 = {wf[j][0], wf[j][1], wf[j][2], wf[j][3]}, b1 = {wf[j][4], wf[j][5], wf[j][6], wf[j][7]};
        acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b0, alo, acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b1, ahi, acc[j], 0, 0, 0);
      }
    }
  };
  for (int t0 = 0; t0 < nsteps; t0 += PASS) {
    if (t0 > 0) {
      __builtin_amdgcn_s_waitcnt(waitcnt_lgkm0_only());  // (the weight scales of the steps before have been read)
      load_x(t0);
      wait_x(std::integral_constant<int, 0>{});
    }
    quantize(std::integral_constant<int, 0>{});
    for_units(t0, [&](auto u_tag) __attribute__((always_inline)) {
      constexpr int u = decltype(u_tag)::value;
      const int begin = t0 + SPU * u;
      step(begin, t0, (u & 1) * SPU, [&]() __attribute__((always_inline)) {
        if constexpr (u + 1 < UNITS)
          if (begin + SPU < nsteps) quantize(std::integral_constant<int, u + 1>{});
      });
      if constexpr (SPU > 1)
        for (int q = 1; q < SPU && begin + q < nsteps; ++q) step(begin + q, t0, (u & 1) * SPU + q, [] {});
    });
  }

  // as gemm_stream_kernel: waves 1..3 leave their partial sums in their own ring, wave 0 adds them in wave order
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  if (wave != 0) {
#pragma unroll
    for (int j = 0; j < NIB; ++j) *reinterpret_cast<acc_t*>(my_ring + j * 1024 + lane * 16) = acc[j];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w)
#pragma unroll
      for (int j = 0; j < NIB; ++j) {
        const acc_t t = *reinterpret_cast<const acc_t*>(smem + w * RING_BYTES + j * 1024 + lane * 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] += t[e];
      }
    if (r16 < p.M) {
#pragma unroll
      for (int j = 0; j < NIB; ++j) {
        const int n = n0 + j * 16 + g * 4;
        if (n < p.N) finish4<KIND, OUT_DT>(p, r16, n, acc[j], out_scale);
      }
    }
  }
}
template <int NIB, int OUT_DT, int IN_DT, int ROWS>
__global__ __launch_bounds__(256) void gemm_stream_quant_kernel(const GemmArgs p) {
  stream_linear_body<KIND_FP8_BLOCK, NIB, OUT_DT, IN_DT, ROWS>(p);
}
template <int KIND, int NIB, int OUT_DT, int IN_DT, int ROWS>
__global__ __launch_bounds__(256) void gemm_stream_tokenquant_kernel(const GemmArgs p) {
  stream_linear_body<KIND, NIB, OUT_DT, IN_DT, ROWS>(p);
}

template <int KIND>
static void launch_stream_linear(GemmArgs& p, int nib, int in_dtype, int out_dtype, hipStream_t st) {
  p.splits = 1;
  p.tiles_m = 1;
  p.tiles_n = (p.N + 16 * nib - 1) / (16 * nib);
  const dim3 grid((uint32_t)p.tiles_n), block(256);
  auto launch = [&](auto nib_tag, auto out_tag, auto in_tag) {
    constexpr int NIB = decltype(nib_tag)::value, OUT_DT = decltype(out_tag)::value, IN_DT = decltype(in_tag)::value;
    auto rows = [&](auto rows_tag) {
      constexpr int ROWS = decltype(rows_tag)::value;
      if constexpr (KIND == KIND_FP8_BLOCK) gemm_stream_quant_kernel<NIB, OUT_DT, IN_DT, ROWS><<<grid, block, 0, st>>>(p);
      else gemm_stream_tokenquant_kernel<KIND, NIB, OUT_DT, IN_DT, ROWS><<<grid, block, 0, st>>>(p);
    };
    if (p.M <= 1) rows(std::integral_constant<int, 1>{});
    else if (p.M <= 2) rows(std::integral_constant<int, 2>{});
    else if (p.M <= 4) rows(std::integral_constant<int, 4>{});
    else rows(std::integral_constant<int, 8>{});
  };
  using one = std::integral_constant<int, 1>;
  using two = std::integral_constant<int, 2>;
  using bf16 = std::integral_constant<int, SGLQ_BF16>;
  using fp16 = std::integral_constant<int, SGLQ_FP16>;
  auto types = [&](auto nib_tag) {
    if (out_dtype == SGLQ_BF16) {
      if (in_dtype == SGLQ_BF16) launch(nib_tag, bf16{}, bf16{});
      else launch(nib_tag, bf16{}, fp16{});
    } else {
      if (in_dtype == SGLQ_BF16) launch(nib_tag, fp16{}, bf16{});
      else launch(nib_tag, fp16{}, fp16{});
    }
  };
  if (nib == 1) types(one{});
  else types(two{});
}

}  // namespace sglq
