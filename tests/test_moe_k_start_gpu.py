"""Grouped GEMMs on weight rows a multiple of 4 KiB apart, whose tiles start at a K block of their own, against the same products in float64: whole
numbers and powers of two, which float32 adds up exactly in any order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (K: one block, fewer than the places to start at, a whole pitch, two of them; experts without rows, rows that end inside a tile)
@pytest.mark.parametrize("k,pitch", [(128, 4096), (384, 4096), (1920, 8192), (4096, 4096), (4224, 8192)])
@pytest.mark.parametrize("tile", [32, 64, 128, 305])  # gemm_kernel's three, the ring's 64 x 128
def test_grouped_k_starts(gpu, k, pitch, tile):
    from sglang_amd import _lib

    print("k starts", k, pitch, tile, flush=True)
    lib = _lib.load()
    n, rows = 272, [33, 0, 1, 70, 131]
    e, m = len(rows), sum(rows)
    g = torch.Generator(device="cuda").manual_seed(k + tile)
    fp8 = lambda *s: torch.randint(-2, 3, s, generator=g, device=gpu).float().to(torch.float8_e4m3fn)
    two_to = lambda *s: 2.0 ** torch.randint(-1, 2, s, generator=g, device=gpu)
    a, w = fp8(m, k), fp8(e, n, pitch)
    sa, sw = two_to(k // 128, m), two_to(e, 3, k // 128)
    offsets = torch.tensor([0] + torch.tensor(rows).cumsum(0).tolist(), dtype=torch.int32, device=gpu)
    sizes = torch.tensor([[r, n, k] for r in rows], dtype=torch.int32, device=gpu)
    out = torch.full((m, n), 3.0, dtype=torch.bfloat16, device=gpu)
    ws = torch.zeros((1 << 16,), dtype=torch.uint8, device=gpu)
    p = lambda t: t.data_ptr()
    lib.sglq_debug_grouped_tile(tile)
    try:
        rc = lib.sglq_fp8_blockwise_scaled_grouped_mm(p(a), k, p(w), pitch, n * pitch, p(sa), 1, m, p(sw), sw.stride(0), 1, sw.stride(1), p(out), n, 0, p(sizes), p(offsets), e, m,
                                                      n, k, p(ws), ws.numel(), _lib.stream_ptr(gpu))
    finally:
        lib.sglq_debug_grouped_tile(0)
    _lib.check(rc, "grouped")
    wide = lambda s: s.double().repeat_interleave(128, dim=-1)
    a64 = a.double() * wide(sa.t())
    for x, r in enumerate(rows):
        own = slice(int(offsets[x]), int(offsets[x]) + r)
        w64 = w[x, :, :k].double() * wide(sw[x]).repeat_interleave(128, dim=0)[:n]
        assert torch.equal(out[own], (a64[own] @ w64.t()).to(torch.bfloat16)), x
