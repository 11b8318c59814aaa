"""The tables of an expert layer and its activations' quantization in one launch against the two one after the other, bit for bit."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# (one slot; steps of 64 slots begun and full; tokens that leave a block half empty; one group, a block's 64 and one more; the most slots a token; no valid id)
@pytest.mark.parametrize("m,topk,e,k,ids_from", [(1, 1, 1, 128, 0), (1, 8, 512, 8192, 0), (65, 1, 7, 8320, -1), (512, 4, 300, 384, -2), (32, 64, 64, 1024, 0), (31, 33, 40, 2048, -9),
                                                 (5, 6, 9, 640, -100)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_tables_with_quantization(gpu, m, topk, e, k, ids_from, dtype):
    from sglang_amd import _lib

    print("tables and quantization", m, topk, e, k, ids_from, dtype, flush=True)
    lib, rows, n, code = _lib.load(), m * topk, 512, 0 if dtype == torch.bfloat16 else 1
    g = torch.Generator(device="cuda").manual_seed(rows + k)
    x = (torch.randn((m, k), generator=g, device=gpu) * 8).to(dtype)
    x[0, :128] = 0
    # ids of nobody on both sides of the experts' range; only such ones
    ids = torch.randint(ids_from, e - ids_from // 2, (m, topk), generator=g, device=gpu, dtype=torch.int32) if ids_from > -100 else torch.full((m, topk), -1, dtype=torch.int32, device=gpu)
    second = ctypes.c_int64(0)
    walk_bytes = lib.sglq_grouped_walk_bytes(e, rows, n, k, ctypes.byref(second))
    p, st = (lambda t: t.data_ptr() if t is not None else None), _lib.stream_ptr(gpu)
    for tile, row_map, walk, once in ((64, False, False, False), (256, True, False, True), (256, True, True, True), (256, True, True, False)):
        if walk and walk_bytes == 0:
            continue

        def state():
            i32 = lambda *shape: torch.full(shape, -7, dtype=torch.int32, device=gpu)
            return [i32(e + 1), i32(e, 3), i32(e, 3), i32(rows), i32(rows) if row_map else None, i32(4 * (rows // tile + e + 1)),
                    torch.full((walk_bytes,), 7, dtype=torch.uint8, device=gpu) if walk else None, torch.full((m if once else rows, k), 9, dtype=torch.uint8, device=gpu),
                    torch.full((k // 128, rows), 5.0, device=gpu)]

        want, got = state(), state()
        tables = lambda t, with_map=row_map: [p(v) for v in t[:4 + with_map]]
        sizes = (rows, e, n, k, tile, rows // tile + e)
        if walk:
            rc = lib.sglq_prepare_moe_layer_walks(p(ids), *tables(want), topk, rows, e, n, k, p(want[5]), p(want[6]), walk_bytes, st)
        elif row_map:
            rc = lib.sglq_prepare_moe_layer_rows(p(ids), *tables(want), topk, *sizes, p(want[5]), st)
        else:
            rc = lib.sglq_prepare_moe_layer(p(ids), *tables(want), *sizes, p(want[5]), st)
        _lib.check(rc, "tables")
        scatter = lib.sglq_per_token_group_quant_fp8_scatter_scales_cm if once else lib.sglq_per_token_group_quant_fp8_scatter_cm
        _lib.check(scatter(p(x), code, p(want[7]), p(want[8]), p(want[3]), m, k, topk, rows, 1e-10, st), "quantization")
        both = lambda t, slots=rows, a_token=topk: lib.sglq_prepare_moe_layer_quant(p(ids), *tables(t, True), a_token, slots, e, n, k, tile, rows // tile + e, p(t[5]), p(t[6]), walk_bytes,
                                                                                    p(x), code, p(t[7]), p(t[8]), once, 1e-10, st)
        _lib.check(both(got), "in one launch")
        for i, (a, b) in enumerate(zip(got, want)):
            assert (a is None and b is None) or torch.equal(a, b), (tile, walk, once, i)
    assert both(got, 2048 + topk) == 1 and both(got, 65, 65) == 1  # more slots than the blocks hold, more of a token
