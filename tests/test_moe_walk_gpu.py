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


# (one segment of slots and several, one expert, experts without rows, more than eight row tiles an expert, columns that end inside a tile)
@pytest.mark.parametrize("m,topk,e,n,k,empty", [(300, 2, 4, 384, 384, True), (515, 3, 4, 512, 640, False), (700, 6, 9, 384, 640, True), (641, 1, 1, 384, 1152, False),
                                                (2500, 8, 32, 384, 1024, False), (4096, 7, 7, 1408, 512, True), (4096, 8, 250, 384, 384, False)])
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
        if row_map_p is not None:
            rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_gathered(p(a), depth, m, p(row_map), *tail(z), p(ps1), p(offsets), 256, *sizes, st)
        else:
            rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_planned(p(a), depth, *tail(z), 256, *sizes, st)
        _lib.check(rc, "in the plan's order")
        assert torch.isfinite(y.float()).all() and torch.equal(y, z)
        assert bool((y[routed:] == 3.0).all())


def test_layers_without_walks(gpu):
    from sglang_amd import _lib

    lib = _lib.load()
    assert lib.sglq_grouped_walk_bytes(32, 32 * 128, 2048, 7168, None) == 0  # 128-row tiles
    assert lib.sglq_grouped_walk_bytes(4, 4096, 256, 7168, None) == 0        # two K blocks
    assert lib.sglq_grouped_walk_bytes(0, 4096, 2048, 7168, None) == 0
