// The activation behind the first GEMM of an expert layer and its quantization in groups of 128, as the GEMMs' epilogues do them: with the expressions of
// silu_mul_group_quant_kernel, bit for bit.
#pragma once
#include "quant_device.h"
#include "sglq_common.h"

namespace sglq {

// 16 rows' accumulators of a wave: gates in acc[0 .. HALF - 1], partners of the same columns behind them, both rounded to 16 bits; two columns to a word of h.
// Returns the largest magnitude, as bits, of the lane's row.
template <int OUT_DT, int HALF, typename acc_t>
SGLQ_DEV uint32_t silu_of_rows(const acc_t (&acc)[2 * HALF], uint32_t (&h)[2 * HALF]) {
  v2us top = {0, 0};
#pragma unroll
  for (int c = 0; c < 2 * HALF; ++c) {
    const acc_t &gate = acc[c >> 1], &partner = acc[HALF + (c >> 1)];
    const int e = 2 * (c & 1);
    h[c] = silu_mul_2x16<OUT_DT>(from_f32_2x16<OUT_DT>(gate[e], gate[e + 1]), from_f32_2x16<OUT_DT>(partner[e], partner[e + 1]));
    top = __builtin_elementwise_max(top, __builtin_bit_cast(v2us, h[c] & 0x7fff7fffu));
  }
  uint32_t m = top.x > top.y ? (uint32_t)top.x : (uint32_t)top.y;
  m = umax(m, (uint32_t)__shfl_xor((int)m, 16));
  return umax(m, (uint32_t)__shfl_xor((int)m, 32));
}

// A group's scale from the waves' maxima, two to a word.
template <int OUT_DT, typename words_t>
SGLQ_DEV float silu_scale(const words_t words, float eps) {
  v2us two = {0, 0};
#pragma unroll
  for (int i = 0; i < (int)(sizeof(words_t) / 4); ++i) {
    const uint32_t word = words[i];  // (a bit cast of a vector's element itself takes the first one)
    two = __builtin_elementwise_max(two, __builtin_bit_cast(v2us, word));
  }
  const uint16_t top = two.x > two.y ? two.x : two.y;
  return div_by(u2f(umax(f2u(to_f32_16<OUT_DT>(top)), f2u(eps))), 448.0f, 1.0f / 448.0f);
}

// The codes of four columns.
template <int OUT_DT>
SGLQ_DEV uint32_t silu_codes(uint32_t h0, uint32_t h1, float y_s, float inv) {
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = quantize_elem<false>(to_f32_16<OUT_DT>((uint16_t)((e < 2 ? h0 : h1) >> (16 * (e & 1)))), y_s, inv, -448.0f, 448.0f);
  return cvt_pk_e4m3<true>(v[2], v[3], cvt_pk_e4m3<false>(v[0], v[1], 0));
}

}  // namespace sglq
