"""The weight-streaming kernels on weights whose rows lie a multiple of 4 KiB apart: a block starts its way round K at a place of its own."""
import ctypes

import pytest
import torch

from oracle import w8a8_oracle as O
from test_gemm_gpu import ATOL, RTOL, rand_i8

pytestmark = pytest.mark.gpu


# K blocks of the four waves: 1 1 1 1 (the smallest K), 2 1 1 1, 3 3 3 2, 8 8 8 8, 17 16 16 16; the last block of weight rows is cut
@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("mnk", [(1, 1032, 512), (16, 2072, 640), (33, 1096, 1408), (8, 4104, 4096), (64, 2056, 8320)])
def test_every_k_block_is_taken_once(gpu, tile, mnk):
    from sglang_amd import _lib

    m, n, k = mnk
    print("stream start", tile, mnk, flush=True)
    lib = _lib.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    pitch = (k + 4095) // 4096 * 4096
    g = torch.Generator().manual_seed(k)

    def rows_apart(w):  # [n, k] as rows `pitch` bytes apart
        wide = torch.zeros((n, pitch), dtype=torch.uint8)
        wide[:, :k] = w.view(torch.uint8)
        return wide.to(gpu)

    # INT8 with unit scales: integer sums below 2^24, exact in float32, so a K block left out or taken twice cannot hide
    a8, w8 = rand_i8((m, k), 1) % 8, rand_i8((n, k), 2) % 8
    ref = a8.float() @ w8.float().t()
    ones_m, ones_n = torch.ones(m, device=gpu), torch.ones(n, device=gpu)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    a_dev, w_dev = a8.to(gpu), rows_apart(w8)
    # block-FP8: the scales of a K block have to come along with it
    af, wf = (torch.randn((m, k), generator=g) * 2).to(torch.float8_e4m3fn), (torch.randn((n, k), generator=g) * 2).to(torch.float8_e4m3fn)
    sfa, sfb = torch.rand((m, k // 128), generator=g) * 0.05 + 0.01, torch.rand(((n + 127) // 128, k // 128), generator=g) * 0.01 + 0.001
    ref_f = O.fp8_blockwise_scaled_mm(af, wf.t(), sfa, sfb.t(), torch.float32, acc_dtype=torch.float64)
    out_f = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    af_dev, wf_dev, dsa, dsb = af.to(gpu), rows_apart(wf), sfa.to(gpu), sfb.to(gpu)
    lib.sglq_debug_force_tile(tile)
    try:
        rc = lib.sglq_int8_scaled_mm(a_dev.data_ptr(), k, w_dev.data_ptr(), pitch, ones_m.data_ptr(), ones_n.data_ptr(), None, out.data_ptr(), n, 0, m, n, k, None, 0, stream)
        assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == f"gemm_stream_kernel<{tile} rows>"
        rc = lib.sglq_fp8_blockwise_scaled_mm(af_dev.data_ptr(), k, wf_dev.data_ptr(), pitch, dsa.data_ptr(), k // 128, 1, dsb.data_ptr(), 1, k // 128,
                                              out_f.data_ptr(), n, 0, m, n, k, None, 0, stream)
        assert rc == 0 and lib.sglq_debug_last_gemm_kernel().decode() == f"gemm_stream_kernel<{tile} rows>"
    finally:
        lib.sglq_debug_force_tile(0)
    assert torch.equal(out.cpu(), ref.to(torch.bfloat16))
    torch.testing.assert_close(out_f.cpu().float(), ref_f, rtol=RTOL, atol=ATOL)
