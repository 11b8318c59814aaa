"""GEMM 1 of an expert layer on 32- and 64-row tiles with the activation behind it (gemm_few_rows_kernel) against GEMM, activation and quantization one after the other, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _both(gpu, rows, n, k, dtype, a, w, sa, sw, tile, gemm=None, nan=False):
    from sglang_amd import _lib

    lib, e, m = _lib.load(), len(rows), sum(rows)
    p, st, code = (lambda t: t.data_ptr()), _lib.stream_ptr(gpu), 0 if dtype == torch.bfloat16 else 1
    ids = torch.repeat_interleave(torch.arange(e, dtype=torch.int32), torch.tensor(rows)).to(gpu)
    i32 = lambda *shape: torch.zeros(shape, dtype=torch.int32, device=gpu)
    plan = i32(4 * (m // tile + e + 1))
    _lib.check(lib.sglq_prepare_moe_layer(p(ids), p(i32(e + 1)), p(i32(e, 3)), p(i32(e, 3)), p(i32(m)), m, e, n, k, tile, m // tile + e, p(plan), st), "tables")
    y = torch.full((m, 2 * n), 3.0, dtype=dtype, device=gpu)
    want_q, q = torch.full((2, m, n), 1, dtype=torch.uint8, device=gpu)
    want_s, s = torch.full((2, n // 128, m), 5.0, device=gpu)
    head = (p(a), k, p(w), w.stride(1), w.stride(0), p(sa), 1, m, p(sw), sw.stride(0), 1, sw.stride(1))
    sizes = (e, m, 2 * n, k, p(plan), plan.numel() * 4)
    lib.sglq_debug_grouped_tile(gemm or tile)
    try:
        _lib.check(lib.sglq_fp8_blockwise_scaled_grouped_mm_planned(*head, p(y), 2 * n, code, tile, *sizes, st), "GEMM")
    finally:
        lib.sglq_debug_grouped_tile(0)
    _lib.check(lib.sglq_silu_and_mul_group_quant_fp8_cm(p(y), code, p(want_q), p(want_s), m, n, 1e-10, st), "activation")
    call = lambda N=2 * n, out=q.data_ptr(), rows=tile: lib.sglq_fp8_blockwise_scaled_grouped_mm_silu_few_rows(*head, out, p(s), code, 1e-10, e, m, N, *sizes[3:], rows, st)
    _lib.check(call(), "in one launch")
    assert call(N=2 * n - 128) == 1 and call(out=q.data_ptr() + 8) == 1 and call(rows=128) == 1
    assert torch.equal(q, want_q)
    torch.testing.assert_close(s, want_s, rtol=0, atol=0, equal_nan=nan)  # (a NaN has no sign to keep)
    return y


# (fewer K blocks than stages; tiles begun, full and one row over; a block's first tile only, several, more than it has lanes for)
@pytest.mark.parametrize("rows,n,k", [([1], 128, 128), ([0, 33, 1, 0, 64, 65, 31], 384, 256), ([32] * 9, 128, 384), ([5, 100] * 30, 1408, 640), ([3] * 40, 1024, 1152),
                                      ([1] * 512, 4224, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile", [32, 64])
def test_activation_on_few_rows(gpu, rows, n, k, dtype, tile):
    print("few rows", len(rows), n, k, dtype, tile, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    e, m = len(rows), sum(rows)
    w = torch.randint(0, 255, (e, 2 * n, k), generator=g, device=gpu, dtype=torch.uint8).clamp_(max=254)
    w = torch.where((w & 127) == 127, 0, w).to(torch.uint8).view(torch.float8_e4m3fn)  # (no NaN)
    sa, sw = torch.rand((k // 128, m), generator=g, device=gpu) + 0.5, torch.rand((e, 2 * n // 128, k // 128), generator=g, device=gpu) * 1e-4 + 1e-5
    _both(gpu, rows, n, k, dtype, torch.randn((m, k), generator=g, device=gpu).to(torch.float8_e4m3fn), w, sa, sw, tile)


@pytest.mark.parametrize("tile", [32, 64])
def test_activation_on_weights_that_start_k_apart(gpu, tile):
    """Weight rows 4 KiB apart, where every tile starts K at a place of its own; whole numbers and powers of two, which float32 adds up exactly in any order."""
    print("few rows, k starts", tile, flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    rows, n, k = [7, 70, 0, 2], 640, 4096
    e, m = len(rows), sum(rows)
    whole = lambda *s: torch.randint(-2, 3, s, generator=g, device=gpu).float().to(torch.float8_e4m3fn)
    two_to = lambda *s: 2.0 ** torch.randint(-9, -7, s, generator=g, device=gpu)
    _both(gpu, rows, n, k, torch.bfloat16, whole(m, k), whole(e, 2 * n, k), two_to(k // 128, m), two_to(e, 2 * n // 128, k // 128), tile)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile", [32, 64])
def test_activation_of_extremes_on_few_rows(gpu, tile, dtype):
    """Rows of infinities, NaN, zeros and values that the 16-bit type cannot hold."""
    print("few rows, extremes", tile, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    rows, n, k = [100, 0, 61, 3], 384, 512
    e, m = len(rows), sum(rows)
    w = torch.randn((e, 2 * n, k), generator=g, device=gpu).to(torch.float8_e4m3fn)
    sa, sw = torch.rand((k // 128, m), generator=g, device=gpu) + 0.5, torch.rand((e, 2 * n // 128, k // 128), generator=g, device=gpu) * 1e-2 + 1e-3
    for i, v in enumerate((float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 1e38, 1e4, 1e-20, 1e-38, -1.0)):
        sa[:, i::13] = v
    y = _both(gpu, rows, n, k, dtype, torch.randn((m, k), generator=g, device=gpu).to(torch.float8_e4m3fn), w, sa, sw, tile, nan=True)
    assert not torch.isfinite(y.float()).all()


# (gemm_kernel's 32 and 64 rows, the ring's 64 x 128; a whole pitch, less than one, more)
@pytest.mark.parametrize("tile,gemm", [(32, 32), (64, 64), (64, 305)])
@pytest.mark.parametrize("k,pitch", [(4096, 4096), (1920, 4096), (4224, 8192)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_sums_in_the_gemm_s_order(gpu, tile, gemm, k, pitch, dtype):
    """Any values on weight rows 4 KiB apart: a tile of gates and partners starts K where the GEMM's tiles of the same columns do."""
    print("few rows, order of the sums", tile, gemm, k, pitch, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(k + tile)
    rows, n = [7, 70, 0, 2], 640
    e, m = len(rows), sum(rows)
    w = torch.randn((e, 2 * n, pitch), generator=g, device=gpu).to(torch.float8_e4m3fn)[:, :, :k]
    sa, sw = torch.rand((k // 128, m), generator=g, device=gpu) + 0.5, torch.rand((e, 2 * n // 128, k // 128), generator=g, device=gpu) * 1e-2 + 1e-3
    _both(gpu, rows, n, k, dtype, torch.randn((m, k), generator=g, device=gpu).to(torch.float8_e4m3fn), w, sa, sw, tile, gemm)


# (tiles of 128 gates: from a quarter round of 256 CUs to one, beyond, from 1.85 rounds, beyond 3.1; all experts and some of them; too few K blocks; 64 rows: from 0.55 rounds,
# around two and above)
@pytest.mark.parametrize("m,topk,e,n,k,rows,activates", [(16, 4, 16, 1536, 1536, 32, 1), (16, 4, 16, 1536, 1408, 32, 0), (8, 8, 32, 1536, 1536, 32, 0), (32, 8, 64, 1024, 1536, 32, 1),
                                                         (60, 8, 64, 2048, 1536, 32, 0), (40, 1, 4, 384, 1536, 32, 0), (5, 3, 41, 1152, 2944, 32, 1),
                                                         (90, 4, 16, 1024, 2048, 32, 1), (122, 4, 16, 1536, 1536, 32, 0), (122, 4, 16, 1536, 1536, 64, 1), (100, 2, 8, 2048, 1536, 64, 0), (480, 4, 60, 1408, 1536, 64, 1), (256, 8, 64, 1024, 1536, 64, 0),
                                                         (1, 8, 16, 3072, 1536, 64, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_layer_of_few_rows(gpu, monkeypatch, m, topk, e, n, k, rows, activates, dtype):
    """What the rule says of tiles of that height, whichever height the layer takes (test_moe_dispatch_gpu.py has what it launches), and the layer's results."""
    import test_moe_tables_gpu as layers

    from sglang_amd import _lib

    assert _lib.load().sglq_grouped_few_rows_activates(e, m, topk, n, k, rows) == activates
    layers.test_layer_host_path(gpu, monkeypatch, m, topk, e, n, k, dtype, torch.float32)


# (weight rows 4 KiB apart: below 12 rows an expert 32-row tiles, above)
@pytest.mark.parametrize("m,topk,e,n", [(16, 4, 16, 1536), (32, 8, 64, 1024), (122, 4, 16, 1536)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_layer_on_weights_4_kib_apart(gpu, monkeypatch, m, topk, e, n, dtype):
    import test_moe_tables_gpu as layers

    layers.test_layer_host_path(gpu, monkeypatch, m, topk, e, n, 4096, dtype, torch.float32)
