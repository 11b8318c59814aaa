"""Which kernel takes a GEMM, at shapes on both sides of a rule's line: the kernel is named and the result compared with the
generic kernel's."""
import ctypes

import pytest
import torch

from test_gemm_ring_gpu import pow2_operands

pytestmark = pytest.mark.gpu
STREAM_32 = "gemm_stream_kernel<32 rows>"
SPLIT_K, SPLIT_K_64 = "gemm_skinny_kernel+splitk_reduce_kernel", "gemm_skinny_kernel<64 columns>+splitk_reduce_kernel"


def operands(gpu, kind, m, n, k):
    """The call of the operator for `kind` on random operands."""
    from sglang_amd.quantization.int8_kernel import w8a8_block_int8_matmul
    from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm, fp8_scaled_mm, int8_scaled_mm
    from sglang_amd.sgl_kernel.gemm import fp8_blockwise_scaled_mm_ue8m0

    a, w, sfa, sfb = pow2_operands(gpu, m, n, k)
    if kind == "pow2":
        return lambda: fp8_blockwise_scaled_mm_ue8m0(a, w.t(), sfa, sfb.t(), torch.bfloat16)
    g = torch.Generator(device=gpu).manual_seed(n)
    if kind == "block":
        sfa, sfb = sfa * torch.rand(sfa.shape, generator=g, device=gpu).t().contiguous().t(), sfb * torch.rand(sfb.shape, generator=g, device=gpu)
        return lambda: fp8_blockwise_scaled_mm(a, w.t(), sfa, sfb.t(), torch.bfloat16)
    sa, sb = torch.rand((m, 1), generator=g, device=gpu) * 0.01 + 1e-3, torch.rand((n, 1), generator=g, device=gpu) * 0.01 + 1e-3
    if kind == "fp8":
        return lambda: fp8_scaled_mm(a, w.t(), sa, sb, torch.bfloat16, None)
    a8, w8 = (torch.randint(-128, 128, s, generator=g, device=gpu, dtype=torch.int8) for s in ((m, k), (n, k)))
    if kind == "i8":
        return lambda: int8_scaled_mm(a8, w8.t(), sa * 0.05, sb, torch.bfloat16, None)
    return lambda: w8a8_block_int8_matmul(a8, w8, sfa * 0.05, sfb * 0.05, [128, 128], torch.bfloat16)


CASES = [
    # 33 to 64 rows, 7/8 of a round of 32-row blocks that start K apart: up to K = 16384, on all of these rows
    ("block", 64, 7424, 16384, STREAM_32),
    ("fp8", 56, 7680, 16384, STREAM_32),
    ("block", 49, 7168, 8192, STREAM_32),
    ("block", 48, 7424, 20480, SPLIT_K),
    ("i8", 40, 7168, 28672, SPLIT_K),
    # few tiles and a long K: a CU's intake bounds gemm_kwave_kernel, the split-K kernel and the ring keep what it had taken;
    # where its tiles fill the chip, or K is short, it stays
    ("i8block", 86, 1216, 7936, SPLIT_K_64),
    ("i8block", 119, 1472, 6784, SPLIT_K_64),
    ("block", 117, 2048, 8192, SPLIT_K_64),
    ("fp8", 201, 1152, 8192, "gemm_ring_kernel"),
    ("fp8", 512, 512, 7168, "gemm_ring_kernel"),
    ("fp8", 128, 2112, 7168, SPLIT_K_64),
    ("block", 630, 1280, 4608, "gemm_kwave_kernel"),
    ("block", 333, 4096, 7040, "gemm_kwave_kernel"),
    ("fp8", 277, 2112, 6400, "gemm_kwave_kernel"),
    ("i8", 506, 1920, 8576, "gemm_kwave_kernel"),
]

PIPE_128 = "gemm_pipe_kernel<128 rows>+splitk_reduce_kernel"
# Power-of-two scales on up to 128 rows: the pipelined 128-row kernel applies them in the MFMA and reads packed words as they are,
# gemm_kwave_kernel and the ring fold them and take packed words expanded by a launch in front
SCALED = [
    (112, 11264, 8192, PIPE_128, PIPE_128),
    (92, 8704, 8192, "gemm_kwave_kernel", PIPE_128),
    (128, 16384, 4096, "gemm_ring_kernel", "gemm_ring_kernel"),
    (96, 11648, 5504, "gemm_kwave_kernel", "gemm_kwave_kernel"),
    (128, 13824, 5120, "gemm_kwave_kernel", "gemm_kwave_kernel"),
]


@pytest.mark.parametrize("m,n,k,kernel,packed_kernel", SCALED)
def test_power_of_two_scales_up_to_128_rows(gpu, m, n, k, kernel, packed_kernel):
    """Same kernel for scales as fp32 and as packed words, unless the expansion costs more than the kernel gains."""
    from sglang_amd import _lib
    from sglang_amd.sgl_kernel import fp8_blockwise_scaled_mm
    from sglang_amd.sgl_kernel.gemm import fp8_blockwise_scaled_mm_ue8m0

    print("selection, power-of-two scales", m, n, k, flush=True)
    lib = _lib.load()
    a, w, sfa, sfb = pow2_operands(gpu, m, n, k)
    plain = fp8_blockwise_scaled_mm(a, w.t(), sfa, sfb.t(), torch.bfloat16)
    out = fp8_blockwise_scaled_mm_ue8m0(a, w.t(), sfa, sfb.t(), torch.bfloat16)
    assert lib.sglq_debug_last_gemm_kernel().decode() == kernel
    assert bool(lib.sglq_debug_last_gemm_hw_scaled()) == (kernel == PIPE_128)
    kb = k // 128
    codes = torch.zeros((m, (kb + 3) // 4 * 4), dtype=torch.uint8, device=gpu)
    codes[:, :kb] = (sfa.contiguous().view(torch.int32) >> 23).to(torch.uint8)
    words = codes.view(torch.int32).t().contiguous()
    scratch, packed_out = torch.empty(64 << 20, dtype=torch.uint8, device=gpu), torch.empty_like(out)
    rc = lib.sglq_fp8_blockwise_scaled_mm_ue8m0_packed(a.data_ptr(), k, w.data_ptr(), k, words.data_ptr(), 1, m, sfb.data_ptr(), 1, kb, packed_out.data_ptr(), n, 0, m, n, k,
                                                       scratch.data_ptr(), scratch.numel(), ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream))
    assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == packed_kernel
    assert bool(lib.sglq_debug_last_gemm_hw_scaled()) == (packed_kernel == PIPE_128)
    for got in (out, packed_out):
        torch.testing.assert_close(got.float(), plain.float(), rtol=1e-2, atol=1e-3 * float(plain.float().std()))


@pytest.mark.parametrize("kind,m,n,k,kernel", CASES)
def test_the_rules_choose(gpu, kind, m, n, k, kernel):
    from sglang_amd import _lib

    print("selection", kind, m, n, k, flush=True)
    lib = _lib.load()
    call = operands(gpu, kind, m, n, k)
    out = call()
    assert lib.sglq_debug_last_gemm_kernel().decode() == kernel
    lib.sglq_debug_force_tile(128)
    try:
        ref = call()
    finally:
        lib.sglq_debug_force_tile(0)
    # (two float32 sums of the same products, each rounded once to bf16: a bf16 step is 2^-8 of the value; what cancels
    # in a sum is bounded by the size of the others)
    assert bool(torch.isfinite(ref).all())
    torch.testing.assert_close(out.float(), ref.float(), rtol=1e-2, atol=1e-3 * float(ref.float().std()))
