"""gemm_ring_kernel (csrc/gemm_ring.h): every tile shape, forced, at the edges of tiles, K blocks and stages."""
import pytest
import torch

from oracle import w8a8_oracle as O
from test_gemm_gpu import ATOL, RTOL, make_block_int8_case, rand_i8

pytestmark = pytest.mark.gpu
RING = 300  # kernel code of configuration 0


@pytest.mark.parametrize("config", range(16))
# one K block; fewer K blocks than stages; a ragged tile of rows and columns past each tile's edge; more tiles than XCDs
@pytest.mark.parametrize("mnk", [(1, 8, 128), (17, 136, 256), (65, 264, 640), (130, 328, 1152), (257, 520, 384)])
def test_ring_kernel_every_tile(gpu, config, mnk):
    from sglang_amd import _lib
    from sglang_amd.quantization.int8_kernel import w8a8_block_int8_matmul
    from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm, fp8_scaled_mm, int8_scaled_mm
    from sglang_amd.sgl_kernel.gemm import fp8_blockwise_scaled_mm_bias

    m, n, k = mnk
    print("ring kernel", config, mnk, flush=True)
    lib = _lib.load()
    lib.sglq_debug_force_tile(RING + config)
    try:
        x8, s8, wq8, ws8 = make_block_int8_case(m, n, k, seed=n + k)
        ref = O.w8a8_block_int8_matmul(x8, wq8, s8, ws8, torch.float32, acc_dtype=torch.float64)
        out = w8a8_block_int8_matmul(x8.to(gpu), wq8.to(gpu), s8.to(gpu), ws8.to(gpu), [128, 128], torch.bfloat16)
        assert lib.sglq_debug_last_gemm_kernel().decode() == "gemm_ring_kernel"
        torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
        g = torch.Generator().manual_seed(m)
        a = (torch.randn((m, k), generator=g) * 2).to(torch.float8_e4m3fn)
        w = (torch.randn((n, k), generator=g) * 2).to(torch.float8_e4m3fn)
        sfa, sfb = torch.rand((m, k // 128), generator=g) * 0.05 + 0.01, torch.rand(((n + 127) // 128, k // 128), generator=g) * 0.01 + 0.001
        bias = (torch.randn(n, generator=g) * 0.1).to(torch.bfloat16)
        ref = O.fp8_blockwise_scaled_mm(a, w.t(), sfa, sfb.t(), torch.float32, acc_dtype=torch.float64)
        args = (a.to(gpu), w.to(gpu).t(), sfa.t().contiguous().to(gpu).t(), sfb.to(gpu).t())
        torch.testing.assert_close(fp8_blockwise_scaled_mm(*args, torch.float16).cpu().float(), ref, rtol=RTOL, atol=ATOL)
        got = fp8_blockwise_scaled_mm_bias(*args, torch.bfloat16, bias.to(gpu)).cpu().float()
        torch.testing.assert_close(got, ref + bias.float(), rtol=RTOL, atol=2 * ATOL)
        for kk in (k, k - 16, k - 112):  # the last K block whole, one chunk short and one chunk long
            a8, w8 = rand_i8((m, kk), 5), rand_i8((n, kk), 6)
            sa, sb = torch.rand((m, 1), generator=g) * 1e-3 + 1e-4, torch.rand((n, 1), generator=g) * 0.01 + 0.001
            ref = O.int8_scaled_mm(a8, w8.t(), sa, sb, torch.bfloat16, bias)
            out = int8_scaled_mm(a8.to(gpu), w8.to(gpu).t(), sa.to(gpu), sb.to(gpu), torch.bfloat16, bias.to(gpu))
            torch.testing.assert_close(out.cpu().float(), ref.float(), rtol=RTOL, atol=ATOL)
            ak, wk = a[:, :kk].contiguous(), w[:, :kk].contiguous()
            ref = O.fp8_scaled_mm(ak, wk.t(), sa, sb, torch.float32, None, acc_dtype=torch.float64)
            out = fp8_scaled_mm(ak.to(gpu), wk.to(gpu).t(), sa.to(gpu), sb.to(gpu), torch.float16, None)
            torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
    finally:
        lib.sglq_debug_force_tile(0)


@pytest.mark.parametrize("mnk", [(333, 512, 1024), (1000, 320, 384), (200, 1088, 1152)])
def test_ring_kernel_power_of_two_scales(gpu, mnk):
    """The scaled-MFMA variant on the tile the rules choose, against the fp32-scale entry point (same sums, another order)."""
    from sglang_amd import _lib
    from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm
    from sglang_amd.sgl_kernel.gemm import fp8_blockwise_scaled_mm_ue8m0

    m, n, k = mnk
    print("ring kernel, power-of-two scales", mnk, flush=True)
    lib = _lib.load()
    g = torch.Generator(device=gpu).manual_seed(m)
    a = (torch.randn((m, k), generator=g, device=gpu) * 2).to(torch.float8_e4m3fn)
    w = (torch.randn((n, k), generator=g, device=gpu) * 2).to(torch.float8_e4m3fn)
    sfa = torch.exp2(torch.randint(-8, -2, (k // 128, m), generator=g, device=gpu).float()).t()
    sfb = torch.exp2(torch.randint(-8, -2, ((n + 127) // 128, k // 128), generator=g, device=gpu).float())
    out = fp8_blockwise_scaled_mm_ue8m0(a, w.t(), sfa, sfb.t(), torch.bfloat16)
    assert lib.sglq_debug_last_gemm_kernel().decode() == "gemm_ring_kernel" and lib.sglq_debug_last_gemm_hw_scaled()
    plain = fp8_blockwise_scaled_mm(a, w.t(), sfa, sfb.t(), torch.bfloat16)
    torch.testing.assert_close(out.float(), plain.float(), rtol=RTOL, atol=ATOL)
