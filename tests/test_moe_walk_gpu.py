"""The walks of an expert layer's GEMMs on 256-row tiles (sglq_prepare_moe_layer_walks) against their definition, and the GEMMs that follow one
against the same GEMMs in the order of the plan, bit for bit."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _tiles(rows):
    """(first row, end row) of the tiles of an expert of `rows` rows: 256 each, the last two sharing what is left in multiples of 32."""
    out, at = [], 0
    while rows - at > 512:
        out.append((at, at + 256))
        at += 256
    if rows - at > 256:
        h = ((rows - at + 1) // 2 + 31) // 32 * 32
        out.append((at, at + h))
        at += h
    if rows > at:
        out.append((at, rows))
    return out


# (one segment of slots and several, one expert, experts without rows, more than eight row tiles an expert, columns that end inside a tile, fewer tiles than XCDs)
@pytest.mark.parametrize("m,topk,e,n,k,empty", [(300, 2, 4, 384, 384, True), (515, 3, 4, 512, 640, False), (700, 6, 9, 384, 640, True), (641, 1, 1, 384, 1152, False),
                                                (2500, 8, 32, 384, 1024, False), (4096, 7, 7, 1408, 512, True), (4096, 8, 250, 384, 384, False), (200, 1, 1, 384, 384, False),
                                                (3, 1, 2, 384, 512, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_walks(gpu, m, topk, e, n, k, empty, dtype):
    from sglang_amd import _lib

    print("walks", m, topk, e, n, k, empty, dtype, flush=True)
    lib = _lib.load()
    rows = m * topk
    g = torch.Generator(device="cuda").manual_seed(rows + e)
    ids = torch.topk(torch.rand((m, e), generator=g, device=gpu) + torch.rand((1, e), generator=g, device=gpu), topk, dim=1)[1].to(torch.int32).contiguous()
    if empty:
        ids[ids == e // 2] = e - 1
        ids[::7, 0] = -1
    second = ctypes.c_int64(0)
    bytes_ = lib.sglq_grouped_walk_bytes(e, rows, n, k, ctypes.byref(second))
    assert bytes_ > second.value > 0
    i32 = lambda *shape: torch.full(shape, 1 << 30, dtype=torch.int32, device=gpu)
    offsets, ps1, ps2, slot_map, row_map, plan = i32(e + 1), i32(e, 3), i32(e, 3), i32(rows), i32(rows), i32(4 * (rows // 256 + e + 1))
    walks = torch.full((bytes_,), 7, dtype=torch.uint8, device=gpu)
    p, st = (lambda t: t.data_ptr()), _lib.stream_ptr(gpu)
    tables = (p(ids), p(offsets), p(ps1), p(ps2), p(slot_map), p(row_map), topk, rows, e, n, k)
    assert lib.sglq_prepare_moe_layer_walks(*tables, p(plan), p(walks), bytes_ - 1, st) == 1
    _lib.check(lib.sglq_prepare_moe_layer_walks(*tables, p(plan), p(walks), bytes_, st), "walks")
    want = [t.clone() for t in (offsets, ps1, ps2, slot_map, row_map)]
    _lib.check(lib.sglq_prepare_moe_layer_rows(*tables, 256, rows // 256 + e, p(plan), st), "tables")
    routed = int(offsets[-1])
    assert all(torch.equal(a, b) for a, b in zip(want[:4], (offsets, ps1, ps2, slot_map))) and torch.equal(want[4][:routed], row_map[:routed])
    off = offsets.tolist()
    out_code = 0 if dtype == torch.bfloat16 else 1
    for width, depth, at, row_map_p in ((2 * n, k, 0, row_map), (k, n, second.value, None)):
        walk = walks[at:].view(torch.int32)[:16 + 4 * (rows // 256 + e) * -(-width // 256)].cpu()
        got = walk[16:16 + 4 * int(walk[0])].view(-1, 4).tolist()
        tiles = {(off[x] + a, off[x] + b, x, c) for x in range(e) for a, b in _tiles(off[x + 1] - off[x]) for c in range(-(-width // 256))}
        assert len(got) == len(tiles) and {tuple(t) for t in got} == tiles
        assert [t[2] for t in got] == sorted(t[2] for t in got)  # expert by expert
        w = torch.randn((e, width, depth), generator=g, device=gpu).to(torch.float8_e4m3fn)
        sw = torch.rand((e, -(-width // 128), depth // 128), generator=g, device=gpu) * 1e-2 + 1e-3
        a = torch.randn((m if row_map_p is not None else rows, depth), generator=g, device=gpu).to(torch.float8_e4m3fn)
        sa = torch.rand((depth // 128, rows), generator=g, device=gpu) + 0.5
        y, z = (torch.full((rows, width), 3.0, dtype=dtype, device=gpu) for _ in range(2))
        tail = lambda o: (p(w), depth, width * depth, p(sa), 1, rows, p(sw), sw.stride(0), 1, sw.stride(1), p(o), width, out_code)
        sizes = (e, rows, width, depth, p(plan), plan.numel() * 4)
        _lib.check(lib.sglq_fp8_blockwise_scaled_grouped_mm_walked(p(a), depth, m, p(row_map) if row_map_p is not None else None, *tail(y), *sizes,
                                                                   p(walks) + at, st), "walked")
        lib.sglq_debug_grouped_tile(256)  # (256 rows where few tiles would take others, too)
        try:
            if row_map_p is not None:
                rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_gathered(p(a), depth, m, p(row_map), *tail(z), p(ps1), p(offsets), 256, *sizes, st)
            else:
                rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_planned(p(a), depth, *tail(z), 256, *sizes, st)
        finally:
            lib.sglq_debug_grouped_tile(0)
        _lib.check(rc, "in the plan's order")
        assert torch.isfinite(y.float()).all() and torch.equal(y, z)
        assert bool((y[routed:] == 3.0).all())
        if row_map_p is not None:
            # ... and with the activation behind it: GEMM, activation and quantization one after the other
            want_q, q = (torch.full((rows, n), 1, dtype=torch.uint8, device=gpu) for _ in range(2))
            want_s, s = (torch.full((n // 128, rows), 5.0, device=gpu) for _ in range(2))
            _lib.check(lib.sglq_silu_and_mul_group_quant_fp8_cm(p(y), out_code, p(want_q), p(want_s), rows, n, 1e-10, st), "activation")
            for name, once in (("gathered", True), ("in place", False)):
                src = a if once else torch.cat([a[row_map[:routed].long()], a[:1].expand(rows - routed, -1)])
                head = (p(src), depth, src.shape[0], p(row_map) if once else None, *tail(q)[:-3])
                _lib.check(lib.sglq_fp8_blockwise_scaled_grouped_mm_silu(*head, p(q), p(s), out_code, 1e-10, *sizes, p(walks) + at, st), name)
                assert torch.equal(q[:routed], want_q[:routed]) and torch.equal(s[:, :routed], want_s[:, :routed]), name
                assert bool((q[routed:] == 1).all()) and bool((s[:, routed:] == 5.0).all())
                q.fill_(1), s.fill_(5.0)


def test_layers_without_walks(gpu):
    from sglang_amd import _lib

    lib = _lib.load()
    assert lib.sglq_grouped_walk_bytes(257, 65536, 2048, 7168, None) == 0  # more experts than the tables' blocks hold
    assert lib.sglq_grouped_walk_bytes(4, 4096, 256, 7168, None) == 0        # two K blocks
    assert lib.sglq_grouped_walk_bytes(0, 4096, 2048, 7168, None) == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_activation_of_extremes(gpu, dtype):
    """Rows of infinities, NaN, zeros and values that the 16-bit type cannot hold through GEMM, activation and quantization: what the three give."""
    from sglang_amd import _lib

    print("extremes", dtype, flush=True)
    lib = _lib.load()
    m, e, n, k = 700, 3, 384, 512
    g = torch.Generator(device="cuda").manual_seed(5)
    ids = torch.randint(0, e, (m, 1), generator=g, device=gpu, dtype=torch.int32)
    second = ctypes.c_int64(0)
    bytes_ = lib.sglq_grouped_walk_bytes(e, m, n, k, ctypes.byref(second))
    i32 = lambda *shape: torch.zeros(shape, dtype=torch.int32, device=gpu)
    offsets, ps1, ps2, slot_map, row_map, plan = i32(e + 1), i32(e, 3), i32(e, 3), i32(m), i32(m), i32(4 * (m // 256 + e + 1))
    walks = torch.zeros(bytes_, dtype=torch.uint8, device=gpu)
    p, st, code = (lambda t: t.data_ptr()), _lib.stream_ptr(gpu), 0 if dtype == torch.bfloat16 else 1
    _lib.check(lib.sglq_prepare_moe_layer_walks(p(ids), p(offsets), p(ps1), p(ps2), p(slot_map), p(row_map), 1, m, e, n, k, p(plan), p(walks), bytes_, st), "walks")
    w = torch.randn((e, 2 * n, k), generator=g, device=gpu).to(torch.float8_e4m3fn)
    sw = torch.rand((e, 2 * n // 128, k // 128), generator=g, device=gpu) * 1e-2 + 1e-3
    a = torch.randn((m, k), generator=g, device=gpu).to(torch.float8_e4m3fn)
    sa = torch.rand((k // 128, m), generator=g, device=gpu) + 0.5
    for i, v in enumerate((float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 1e38, 1e4, 1e-20, 1e-38, -1.0)):
        sa[:, i::13] = v
    y = torch.zeros((m, 2 * n), dtype=dtype, device=gpu)
    tail = (p(w), k, 2 * n * k, p(sa), 1, m, p(sw), sw.stride(0), 1, sw.stride(1))
    sizes = (e, m, 2 * n, k, p(plan), plan.numel() * 4)
    _lib.check(lib.sglq_fp8_blockwise_scaled_grouped_mm_walked(p(a), k, m, None, *tail, p(y), 2 * n, code, *sizes, p(walks), st), "walked")
    (want_q, q), (want_s, s) = torch.zeros((2, m, n), dtype=torch.uint8, device=gpu), torch.zeros((2, n // 128, m), device=gpu)
    _lib.check(lib.sglq_silu_and_mul_group_quant_fp8_cm(p(y), code, p(want_q), p(want_s), m, n, 1e-10, st), "activation")
    _lib.check(lib.sglq_fp8_blockwise_scaled_grouped_mm_silu(p(a), k, m, None, *tail, p(q), p(s), code, 1e-10, *sizes, p(walks), st), "in one launch")
    assert not torch.isfinite(y.float()).all()
    assert torch.equal(q, want_q)
    torch.testing.assert_close(s, want_s, rtol=0, atol=0, equal_nan=True)  # (a NaN has no sign to keep)


# (the row tiles that the layer's sizes choose; on 256 rows the activation in GEMM 1 up to 128 rows an expert and from 96 tiles' worth, 24 x 3 and 35 x 3 here;
# 0: each GEMM's own, below 12 rows an expert and on intermediate sizes without a walk)
@pytest.mark.parametrize("m,topk,e,n,k,tile", [(900, 6, 6, 384, 512, 256), (1400, 6, 6, 384, 512, 256), (1400, 2, 5, 384, 1024, 256), (300, 8, 32, 1024, 1024, 256),
                                               (121, 3, 24, 384, 1152, 32), (1326, 1, 9, 384, 2048, 64), (600, 2, 5, 2048, 1024, 128), (95, 4, 32, 384, 1664, 0),
                                               (900, 6, 6, 256, 512, 0)])
def test_layer(gpu, monkeypatch, m, topk, e, n, k, tile):
    import test_moe_tables_gpu as layers

    from sglang_amd import _lib

    assert _lib.load().sglq_grouped_layer_rows(e, m, topk, n, k) == tile
    layers.test_layer_host_path(gpu, monkeypatch, m, topk, e, n, k, torch.bfloat16, torch.float32)


# (fp16, where neither the layer nor the operators take 128-row tiles, whose last step rounds once)
@pytest.mark.parametrize("m,topk,e,n,k", [(900, 6, 6, 384, 512), (1400, 6, 6, 384, 512), (1400, 2, 5, 384, 1024), (121, 3, 24, 384, 1152), (1326, 1, 9, 384, 2048)])
def test_layer_of_halves(gpu, monkeypatch, m, topk, e, n, k):
    import test_moe_tables_gpu as layers

    layers.test_layer_host_path(gpu, monkeypatch, m, topk, e, n, k, torch.float16, torch.float32)
