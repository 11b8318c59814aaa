"""gemm_kwave_kernel (csrc/gemm_kwave.h): every tile shape, forced, at the edges of tiles, rings and the waves' shares of K."""
import pytest
import torch

from oracle import w8a8_oracle as O
from test_gemm_gpu import ATOL, RTOL, make_block_int8_case, rand_i8

pytestmark = pytest.mark.gpu
KWAVE = 270  # kernel code of configuration 0
IN_PLACE_ONLY = (5, 9, 10)  # tile shapes that the block-scaled kinds do not have


# fewer K blocks than waves; five: one wave has two; tiles cut by M and N; thirteen to forty-one: the ring's positions repeat
@pytest.mark.parametrize("config", range(11))
@pytest.mark.parametrize("mnk", [(1, 8, 128), (17, 72, 256), (65, 136, 640), (130, 264, 1664), (225, 200, 5248)])
def test_kwave_kernel_every_tile(gpu, config, mnk):
    from sglang_amd import _lib
    from sglang_amd.quantization.int8_kernel import w8a8_block_int8_matmul
    from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm, fp8_scaled_mm, int8_scaled_mm
    from sglang_amd.sgl_kernel.gemm import fp8_blockwise_scaled_mm_bias

    m, n, k = mnk
    print("kwave kernel", config, mnk, flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(m)
    a = (torch.randn((m, k), generator=g) * 2).to(torch.float8_e4m3fn)
    w = (torch.randn((n, k), generator=g) * 2).to(torch.float8_e4m3fn)
    bias = (torch.randn(n, generator=g) * 0.1).to(torch.bfloat16)
    lib.sglq_debug_force_tile(KWAVE + config)
    try:
        if config not in IN_PLACE_ONLY:
            x8, s8, wq8, ws8 = make_block_int8_case(m, n, k, seed=n + k)
            ref = O.w8a8_block_int8_matmul(x8, wq8, s8, ws8, torch.float32, acc_dtype=torch.float64)
            out = w8a8_block_int8_matmul(x8.to(gpu), wq8.to(gpu), s8.to(gpu), ws8.to(gpu), [128, 128], torch.bfloat16)
            assert lib.sglq_debug_last_gemm_kernel().decode() == "gemm_kwave_kernel"
            torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
            sfa, sfb = torch.rand((m, k // 128), generator=g) * 0.05 + 0.01, torch.rand(((n + 127) // 128, k // 128), generator=g) * 0.01 + 0.001
            ref = O.fp8_blockwise_scaled_mm(a, w.t(), sfa, sfb.t(), torch.float32, acc_dtype=torch.float64)
            args = (a.to(gpu), w.to(gpu).t(), sfa.t().contiguous().to(gpu).t(), sfb.to(gpu).t())
            torch.testing.assert_close(fp8_blockwise_scaled_mm(*args, torch.float16).cpu().float(), ref, rtol=RTOL, atol=ATOL)
            got = fp8_blockwise_scaled_mm_bias(*args, torch.bfloat16, bias.to(gpu)).cpu().float()
            torch.testing.assert_close(got, ref + bias.float(), rtol=RTOL, atol=2 * ATOL)
        a8, w8 = rand_i8((m, k), 5), rand_i8((n, k), 6)
        sa, sb = torch.rand((m, 1), generator=g) * 1e-3 + 1e-4, torch.rand((n, 1), generator=g) * 0.01 + 0.001
        ref = O.int8_scaled_mm(a8, w8.t(), sa, sb, torch.bfloat16, bias)
        out = int8_scaled_mm(a8.to(gpu), w8.to(gpu).t(), sa.to(gpu), sb.to(gpu), torch.bfloat16, bias.to(gpu))
        assert lib.sglq_debug_last_gemm_kernel().decode() == "gemm_kwave_kernel"
        torch.testing.assert_close(out.cpu().float(), ref.float(), rtol=RTOL, atol=ATOL)
        ref = O.fp8_scaled_mm(a, w.t(), sa, sb, torch.float32, None, acc_dtype=torch.float64)
        out = fp8_scaled_mm(a.to(gpu), w.to(gpu).t(), sa.to(gpu), sb.to(gpu), torch.float16, None)
        torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
    finally:
        lib.sglq_debug_force_tile(0)


def test_kwave_kernel_reads_strided_operands(gpu):
    """Rows longer than K, row-major activation scales, an output that is part of a wider one."""
    import ctypes

    from sglang_amd import _lib

    m, n, k, pad = 200, 328, 1152, 256
    print("kwave kernel, strides", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(3)
    a = (torch.randn((m, k + pad), generator=g) * 2).to(torch.float8_e4m3fn)
    w = (torch.randn((n, k + pad), generator=g) * 2).to(torch.float8_e4m3fn)
    sfa, sfb = torch.rand((m, k // 128), generator=g) * 0.05 + 0.01, torch.rand(((n + 127) // 128, k // 128), generator=g) * 0.01 + 0.001
    ref = O.fp8_blockwise_scaled_mm(a[:, :k].contiguous(), w[:, :k].contiguous().t(), sfa, sfb.t(), torch.float32, acc_dtype=torch.float64)
    out = torch.full((m, n + 64), 7.0, dtype=torch.bfloat16, device=gpu)
    da, dw, dsa, dsb = a.to(gpu), w.to(gpu), sfa.to(gpu), sfb.to(gpu)
    lib.sglq_debug_force_tile(KWAVE + 2)
    try:
        rc = lib.sglq_fp8_blockwise_scaled_mm(da.data_ptr(), k + pad, dw.data_ptr(), k + pad, dsa.data_ptr(), k // 128, 1, dsb.data_ptr(), 1, k // 128,
                                              out.data_ptr(), n + 64, 0, m, n, k, None, 0, ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream))
    finally:
        lib.sglq_debug_force_tile(0)
    assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == "gemm_kwave_kernel"
    torch.testing.assert_close(out[:, :n].cpu().float(), ref, rtol=RTOL, atol=ATOL)
    assert bool((out[:, n:] == 7.0).all())


# the entry points that only the tile's epilogue or a launch in front sets apart; both output types, M and N cut
@pytest.mark.parametrize("config", [c for c in range(11) if c not in IN_PLACE_ONLY])
def test_kwave_kernel_block_int8_bias_and_packed_scales(gpu, config):
    import ctypes

    from sglang_amd import _lib
    from sglang_amd.quantization.int8_kernel import w8a8_block_int8_matmul
    from test_gemm_ring_gpu import pow2_operands

    m, n, k = 130, 264, 1408
    print("kwave kernel, block-INT8 bias, packed scales", config, flush=True)
    lib = _lib.load()
    x8, s8, wq8, ws8 = make_block_int8_case(m, n, k, seed=config)
    a, w, sfa, sfb = pow2_operands(gpu, m, n, k)
    kb = k // 128
    codes = torch.zeros((m, (kb + 3) // 4 * 4), dtype=torch.uint8)
    codes[:, :kb] = (sfa.cpu().contiguous().view(torch.int32) >> 23).to(torch.uint8)
    words, scratch = codes.view(torch.int32).t().contiguous().to(gpu), torch.empty(4 * m * kb + 4096, dtype=torch.uint8, device=gpu)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    lib.sglq_debug_force_tile(KWAVE + config)
    try:
        for dtype in (torch.bfloat16, torch.float16):
            bias = (torch.randn(n, generator=torch.Generator().manual_seed(config)) * 0.1).to(dtype)
            ref = O.w8a8_block_int8_matmul(x8, wq8, s8, ws8, torch.float32, acc_dtype=torch.float64) + bias.float()
            got = w8a8_block_int8_matmul(x8.to(gpu), wq8.to(gpu), s8.to(gpu), ws8.to(gpu), [128, 128], dtype, bias=bias.to(gpu))
            assert lib.sglq_debug_last_gemm_kernel().decode() == "gemm_kwave_kernel"
            torch.testing.assert_close(got.cpu().float(), ref, rtol=RTOL, atol=2 * ATOL)  # (rounded twice: the product, then with the bias)
        rc = lib.sglq_fp8_blockwise_scaled_mm_ue8m0_packed(a.data_ptr(), k, w.data_ptr(), k, words.data_ptr(), 1, m, sfb.data_ptr(), 1, kb, out.data_ptr(), n, 0, m, n, k,
                                                           scratch.data_ptr(), scratch.numel(), ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream))
        assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == "gemm_kwave_kernel" and not lib.sglq_debug_last_gemm_hw_scaled()
    finally:
        lib.sglq_debug_force_tile(0)
    ref = O.fp8_blockwise_scaled_mm(a.cpu(), w.cpu().t(), sfa.cpu(), sfb.cpu().t(), torch.float32, acc_dtype=torch.float64)
    torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
