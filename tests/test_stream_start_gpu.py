"""Weights whose rows lie a multiple of 4 KiB apart: each tile of them starts its way round K at a place of its own."""
import ctypes

import pytest
import torch

from oracle import w8a8_oracle as O
from test_gemm_gpu import ATOL, RTOL, rand_i8
from test_gemm_ring_gpu import pow2_operands

pytestmark = pytest.mark.gpu


STREAM = {16: "gemm_stream_kernel<16 rows>", 32: "gemm_stream_kernel<32 rows>"}
SHARED = {64: "gemm_skinny_kernel", 66: "gemm_skinny_kernel<64 columns>", 270: "gemm_kwave_kernel", 276: "gemm_kwave_kernel", 300: "gemm_ring_kernel",
          304: "gemm_ring_kernel", 314: "gemm_ring_kernel"}  # the ring's take one, two and four K blocks a stage


# K blocks of the four waves: 1 1 1 1 (the smallest K), 2 1 1 1, 3 3 3 2, 8 8 8 8, 17 16 16 16; the last block of weight rows is cut.
# The kernels whose blocks share activation tiles take 48 weight rows to an activation row; odd numbers of K blocks, one that is cut.
CASES = [(t, s) for t in STREAM for s in [(1, 1032, 512), (16, 2072, 640), (33, 1096, 1408), (8, 4104, 4096), (64, 2056, 8320)]]
CASES += [(t, s) for t in SHARED for s in ([(17, 1032, 640)] if t != 66 else []) + [(40, 2072, 1408), (33, 2056, 8320)]]
CASES += [(t, (20, 1000, 1008)) for t in (300, 304, 314)]


def rows_apart(w, gpu):
    """[n, k] of bytes as rows the next multiple of 4 KiB apart."""
    wide = torch.zeros((w.shape[0], (w.shape[1] + 4095) // 4096 * 4096), dtype=torch.uint8)
    wide[:, : w.shape[1]] = w.view(torch.uint8)
    return wide.to(gpu)


@pytest.mark.parametrize("tile,mnk", CASES)
def test_every_k_block_is_taken_once(gpu, tile, mnk):
    from sglang_amd import _lib

    m, n, k = mnk
    kernel = {**STREAM, **SHARED}[tile]
    print("start of K", tile, mnk, flush=True)
    lib = _lib.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    lib.sglq_debug_force_tile(tile)
    lib.sglq_debug_force_splits(1)
    try:
        # INT8 with unit scales: integer sums below 2^24, exact in float32, so a K block left out or taken twice cannot hide
        a8, w8 = rand_i8((m, k), 1) % 8, rand_i8((n, k), 2) % 8
        a, w, one_m, one_n = a8.to(gpu), rows_apart(w8, gpu), torch.ones(m, device=gpu), torch.ones(n, device=gpu)
        out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
        rc = lib.sglq_int8_scaled_mm(a.data_ptr(), k, w.data_ptr(), w.stride(0), one_m.data_ptr(), one_n.data_ptr(), None, out.data_ptr(), n, 0, m, n, k, None, 0, stream)
        assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == kernel
        assert torch.equal(out.cpu(), (a8.float() @ w8.float().t()).to(torch.bfloat16))
        if k % 128:
            return
        # block-FP8: the scales of a K block have to come along with it
        g, kb = torch.Generator().manual_seed(k), k // 128
        af, wf = (torch.randn((m, k), generator=g) * 2).to(torch.float8_e4m3fn), (torch.randn((n, k), generator=g) * 2).to(torch.float8_e4m3fn)
        sfa, sfb = torch.rand((m, kb), generator=g) * 0.05 + 0.01, torch.rand(((n + 127) // 128, kb), generator=g) * 0.01 + 0.001
        ref = O.fp8_blockwise_scaled_mm(af, wf.t(), sfa, sfb.t(), torch.float32, acc_dtype=torch.float64)
        a, w, dsa, dsb = af.to(gpu), rows_apart(wf, gpu), sfa.to(gpu), sfb.to(gpu)
        rc = lib.sglq_fp8_blockwise_scaled_mm(a.data_ptr(), k, w.data_ptr(), w.stride(0), dsa.data_ptr(), kb, 1, dsb.data_ptr(), 1, kb, out.data_ptr(), n, 0, m, n, k, None, 0, stream)
        assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == kernel
        torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
    finally:
        lib.sglq_debug_force_tile(0)
        lib.sglq_debug_force_splits(0)


@pytest.mark.parametrize("config", [0, 4, 14])  # two, one and four K blocks a stage
def test_packed_scales_follow_the_k_blocks(gpu, config):
    """Scales as words of four K blocks' exponent bytes: the byte is the K block's, wherever the tile starts."""
    from sglang_amd import _lib

    m, n, k = 130, 6248, 1408  # (more than 128 rows: scales in the matrix instruction)
    print("start of K, packed scales", config, flush=True)
    lib = _lib.load()
    a, w, sfa, sfb = pow2_operands(gpu, m, n, k)
    kb = k // 128
    ref = O.fp8_blockwise_scaled_mm(a.cpu(), w.cpu().t(), sfa.cpu(), sfb.cpu().t(), torch.float32, acc_dtype=torch.float64)
    codes = torch.zeros((m, (kb + 3) // 4 * 4), dtype=torch.uint8)
    codes[:, :kb] = (sfa.cpu().contiguous().view(torch.int32) >> 23).to(torch.uint8)
    words, wide = codes.view(torch.int32).t().contiguous().to(gpu), rows_apart(w.cpu(), gpu)
    scratch = torch.empty(4 * m * kb + 4096, dtype=torch.uint8, device=gpu)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    lib.sglq_debug_force_tile(300 + config)
    try:
        rc = lib.sglq_fp8_blockwise_scaled_mm_ue8m0_packed(a.data_ptr(), k, wide.data_ptr(), wide.stride(0), words.data_ptr(), 1, m, sfb.data_ptr(), 1, kb, out.data_ptr(), n, 0,
                                                           m, n, k, scratch.data_ptr(), scratch.numel(), ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream))
        assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == "gemm_ring_kernel" and lib.sglq_debug_last_gemm_hw_scaled()
    finally:
        lib.sglq_debug_force_tile(0)
    torch.testing.assert_close(out.cpu().float(), ref, rtol=RTOL, atol=ATOL)
