"""cutlass_fused_experts_fp8 with the reference's argument list and call sequence
(python/sglang/srt/layers/moe/cutlass_moe.py:30-222), on the HIP operators."""

from __future__ import annotations

import torch

from .. import _lib
from .._lib import native
from ..sgl_kernel import apply_shuffle_mul_sum, fp8_blockwise_scaled_grouped_mm, prepare_moe_input
from ..sgl_kernel.moe import per_token_group_quant_fp8_to_expert_rows, silu_and_mul_per_token_group_quant_fp8


def cutlass_fused_experts_fp8(
    a: torch.Tensor,
    w1_q: torch.Tensor,
    w2_q: torch.Tensor,
    w1_scale: torch.Tensor,
    w2_scale: torch.Tensor,
    topk_weights: torch.Tensor,
    topk_ids: torch.Tensor,
    a1_strides: torch.Tensor,
    c1_strides: torch.Tensor,
    a2_strides: torch.Tensor,
    c2_strides: torch.Tensor,
    workspace: torch.Tensor,
    a_ptrs: torch.Tensor,
    b_ptrs: torch.Tensor,
    out_ptrs: torch.Tensor,
    a_scales_ptrs: torch.Tensor,
    b_scales_ptrs: torch.Tensor,
    expert_offsets: torch.Tensor,
    problem_sizes1: torch.Tensor,
    problem_sizes2: torch.Tensor,
    use_fp8_blockscale: bool = True,
) -> torch.Tensor:
    """MoE expert layer with SiLU-gated FFNs, FP8 weights with 128 x 128 block scales and
    per-token-group-128 FP8 activations (cutlass_moe.py:30-222).

    a [m, k] half / bfloat16; w1_q [E, k, 2 n] and w2_q [E, n, k] e4m3fn, every expert's slice
    column-major (the transposed views of the [E, 2 n, k] / [E, k, n] weights); w1_scale
    [E, k/128, 2 n/128] and w2_scale [E, n/128, k/128] fp32 with any strides; topk_weights and
    topk_ids [m, topk]; expert_offsets [E + 1] and problem_sizes1/2 [E, 3] int32 are filled here.
    Steps: routing tables; activations quantized once per token and written (codes and
    scales) to their expert-major rows; grouped GEMM 1; SiLU-and-multiply fused with the second
    quantization; grouped GEMM 2; weighted sum back into token order.  No per-expert transpose pass is needed: the
    C++ host path writes the activation scales column-major over all rows (a K block's scales of 64 rows are then one
    load; with many rows an expert it writes the codes once, in token order, and GEMM 1 gathers them), the steps below keep them K-major, the branch the reference takes for SM100 (:160-162,194-196)."""
    assert use_fp8_blockscale, "Only support fp8 blockscale for now"
    assert topk_weights.shape == topk_ids.shape, "topk shape mismatch"
    assert w1_q.dtype == torch.float8_e4m3fn
    assert w2_q.dtype == torch.float8_e4m3fn
    assert a.shape[1] == w1_q.shape[1], "Hidden size mismatch w1"
    assert w1_q.shape[2] == w2_q.shape[1] * 2, "Hidden size mismatch w2"
    assert w1_q.shape[0] == w2_q.shape[0], "Expert number mismatch"
    assert w1_q.shape[0] == w1_scale.shape[0], "w1 scales expert number mismatch"
    assert w1_q.shape[0] == w2_scale.shape[0], "w2 scales expert number mismatch"
    assert a.dtype in [torch.half, torch.bfloat16], "Invalid output dtype"
    _lib.load()  # (binds the host path: a process's first layer takes its tiles too, and so gives every later one's bits)
    result = native.experts(a, w1_q, w2_q, w1_scale, w2_scale, topk_weights, topk_ids, expert_offsets, problem_sizes1, problem_sizes2)
    if result is not None:
        return result

    out_dtype = a.dtype
    num_experts = w1_q.size(0)
    m = a.size(0)
    k = w1_q.size(1)
    n = w2_q.size(1)
    topk = topk_ids.size(1)
    device = a.device

    a_map = torch.empty((topk_ids.numel()), dtype=torch.int32, device=device)
    # slots whose expert id is outside [0, E) are routed nowhere: -1 makes the combine skip them
    c_map = torch.full((topk_ids.numel(),), -1, dtype=torch.int32, device=device)
    prepare_moe_input(topk_ids, expert_offsets, problem_sizes1, problem_sizes2, a_map, c_map, num_experts, n, k)

    # sglang_per_token_group_quant_fp8(a, 128) and the two shuffle_rows(., a_map, .) calls
    # (cutlass_moe.py:156-158) in one kernel: every token is quantized once and written to its rows
    rep_a_q, rep_a1_scales = per_token_group_quant_fp8_to_expert_rows(a, c_map, topk, 128)

    c1 = torch.empty((m * topk, n * 2), device=device, dtype=out_dtype)
    c2 = torch.empty((m * topk, k), device=device, dtype=out_dtype)
    a_sf_layout = torch.empty((num_experts, 5), device=device, dtype=torch.int)
    w_sf_layout = torch.empty((num_experts, 5), device=device, dtype=torch.int)

    fp8_blockwise_scaled_grouped_mm(
        c1, a_ptrs, b_ptrs, out_ptrs, a_scales_ptrs, b_scales_ptrs, rep_a_q, w1_q, rep_a1_scales, w1_scale,
        a1_strides, a1_strides, c1_strides, a_sf_layout, w_sf_layout, problem_sizes1, expert_offsets[:-1], workspace)

    # silu_and_mul(c1, intermediate) and sglang_per_token_group_quant_fp8(intermediate, 128)
    # (cutlass_moe.py:187-194) in one kernel with the same codes and scales
    intermediate_q, a2_scale = silu_and_mul_per_token_group_quant_fp8(c1, 128)

    fp8_blockwise_scaled_grouped_mm(
        c2, a_ptrs, b_ptrs, out_ptrs, a_scales_ptrs, b_scales_ptrs, intermediate_q, w2_q, a2_scale, w2_scale,
        a2_strides, a2_strides, c2_strides, a_sf_layout, w_sf_layout, problem_sizes2, expert_offsets[:-1], workspace)

    result = torch.empty((m, k), device=device, dtype=out_dtype)
    apply_shuffle_mul_sum(c2, result, c_map, topk_weights.to(out_dtype))
    return result
