"""The grouped GEMM on gemm_ring_kernel's 64 x 128 tiles: few and uneven experts, empty ones, ragged columns and K; and the
column-major scale outputs of the expert layer's two quantization kernels."""
import pytest
import torch

from test_moe_gpu import run_grouped

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def grouped_case(gpu, rows, n, k, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    e, total = len(rows), sum(rows)
    cuts = torch.tensor([0] + rows).cumsum(0)
    a = (torch.randn((total, k), generator=g, device=gpu) * 2).to(FP8)
    b = torch.randn((e, n, k), generator=g, device=gpu).to(FP8)
    sa = torch.rand((total, k // 128), generator=g, device=gpu) * 0.01 + 0.001
    sb = torch.rand((e, k // 128, (n + 127) // 128), generator=g, device=gpu) * 0.01 + 0.001
    case = dict(a=a, b=b.transpose(1, 2), scales_a=sa, scales_b=sb, problem_sizes=torch.tensor([[r, n, k] for r in rows], dtype=torch.int32),
                expert_offsets=cuts[:-1].to(torch.int32))
    return case, cuts, b, sb


@pytest.mark.parametrize("rows", [[1], [0, 3, 0, 5], [64, 1, 65, 0, 130], [17] * 9])
@pytest.mark.parametrize("nk", [(128, 128), (136, 1152), (1024, 384)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_grouped_ring_tiles(gpu, rows, nk, dtype):
    from sglang_amd import _lib

    n, k = nk
    n += -n % 128  # the operator's scale layout is whole blocks of columns
    print("grouped ring tiles", rows, n, k, dtype, flush=True)
    lib = _lib.load()
    case, cuts, b, sb = grouped_case(gpu, rows, n, k, seed=sum(rows) + n)
    lib.sglq_debug_grouped_tile(305)
    try:
        out = run_grouped(gpu, case, dtype)
        assert lib.sglq_debug_last_gemm_kernel().decode().endswith("gemm_ring_kernel<grouped>")
    finally:
        lib.sglq_debug_grouped_tile(0)
    for x, r in enumerate(rows):
        sl = slice(int(cuts[x]), int(cuts[x + 1]))
        a = case["a"][sl].float() * case["scales_a"][sl].repeat_interleave(128, dim=1)
        w = b[x].float() * sb[x].t().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)[:n]
        torch.testing.assert_close(out[sl].float(), a @ w.t(), rtol=1e-2, atol=1e-2)


# an expert's last two 256-row tiles share what is left in multiples of 32 rows, five to eight per half tile: a single tile of each
# height, two of them around each change of height, whole tiles in front of them; then the same without a next expert's rows behind
@pytest.mark.parametrize("rows", [[1, 33, 160, 161, 192, 193, 224, 225, 256], [257, 288, 320, 321, 384, 385, 448, 449, 511], [512, 513, 0, 769, 600], [150], [417]])
@pytest.mark.parametrize("nk", [(384, 384), (512, 1152)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_grouped_256_row_tiles_share_the_last_rows(gpu, rows, nk, dtype):
    from sglang_amd import _lib

    n, k = nk
    print("grouped 256-row tiles", rows, n, k, dtype, flush=True)
    lib = _lib.load()
    case, cuts, b, sb = grouped_case(gpu, rows, n, k, seed=sum(rows) + n)
    lib.sglq_debug_grouped_tile(256)
    try:
        out = run_grouped(gpu, case, dtype)
        assert lib.sglq_debug_last_gemm_kernel().decode().endswith("gemm_pipe_kernel<grouped>")
    finally:
        lib.sglq_debug_grouped_tile(0)
    for x, r in enumerate(rows):
        sl = slice(int(cuts[x]), int(cuts[x + 1]))
        a = case["a"][sl].float() * case["scales_a"][sl].repeat_interleave(128, dim=1)
        w = b[x].float() * sb[x].t().repeat_interleave(128, dim=0).repeat_interleave(128, dim=1)[:n]
        torch.testing.assert_close(out[sl].float(), a @ w.t(), rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,d", [(1, 128), (15, 384), (33, 256), (100, 1152)])
def test_column_major_scales(gpu, dtype, m, d):
    """Same codes as the row-major entry points, the scales transposed; rows nobody names untouched."""
    from sglang_amd import _lib

    lib = _lib.load()
    code, st = _lib.DTYPE_CODE[dtype], torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=gpu).manual_seed(m)
    x = torch.randn((m, 2 * d), generator=g, device=gpu).to(dtype)
    got = []
    for fn, shape in ((lib.sglq_silu_and_mul_group_quant_fp8, (m, d // 128)), (lib.sglq_silu_and_mul_group_quant_fp8_cm, (d // 128, m))):
        q, s = torch.zeros((m, d), dtype=torch.uint8, device=gpu), torch.zeros(shape, device=gpu)
        assert fn(x.data_ptr(), code, q.data_ptr(), s.data_ptr(), m, d, 1e-10, st) == 0
        got.append((q, s))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1].t())
    topk, rows = 3, 2 * m + 5
    xs = x[:, :d].contiguous()
    slots = torch.randperm(rows + m, generator=g, device=gpu)[: m * topk].to(torch.int32) - 2  # some outside, some rows nobody's
    got = []
    for fn, shape in ((lib.sglq_per_token_group_quant_fp8_scatter, (rows, d // 128)), (lib.sglq_per_token_group_quant_fp8_scatter_cm, (d // 128, rows))):
        q, s = torch.full((rows, d), 7, dtype=torch.uint8, device=gpu), torch.full(shape, -1.0, device=gpu)
        assert fn(xs.data_ptr(), code, q.data_ptr(), s.data_ptr(), slots.data_ptr(), m, d, topk, rows, 1e-10, st) == 0
        got.append((q, s))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1].t())
