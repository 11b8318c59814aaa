"""The expert layer's tables in one launch (sglq_prepare_moe_layer) against the oracle's at the edges of what it
takes, its tile plan against the definition, and the layer's host path against the same layer called
operator by operator, bit for bit."""
import pytest
import torch

from oracle import w8a8_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots,experts,tile", [(1, 1, 64), (64, 3, 16), (65, 32, 64), (1024, 33, 128), (1025, 256, 16), (20000, 32, 256), (32767, 512, 64),
                                                (32768, 2, 256)])
def test_tables_and_plan(gpu, slots, experts, tile):
    from sglang_amd import _lib

    print("tables", slots, experts, tile, flush=True)
    g = torch.Generator().manual_seed(slots + experts)
    ids = torch.randint(0, experts, (slots, 1), generator=g, dtype=torch.int32)
    if slots > 16:
        ids[3], ids[7] = -1, experts  # routed to nobody
        ids[slots // 2:slots // 2 + slots // 4] = ids[0]  # a crowded expert
    n, k = 384, 512
    want = O.prepare_moe_input(ids, experts, n, k)
    i32 = lambda *shape: torch.full(shape, -7, dtype=torch.int32, device=gpu)
    offsets, ps1, ps2, c_map = i32(experts + 1), i32(experts, 3), i32(experts, 3), i32(slots)
    max_tiles = slots // tile + experts
    plan = i32(4 * (max_tiles + 1))
    rc = _lib.load().sglq_prepare_moe_layer(ids.to(gpu).data_ptr(), offsets.data_ptr(), ps1.data_ptr(), ps2.data_ptr(), c_map.data_ptr(), slots, experts,
                                            n, k, tile, max_tiles, plan.data_ptr(), _lib.stream_ptr(gpu))
    _lib.check(rc, "prepare_moe_layer")
    assert torch.equal(offsets.cpu(), want[0]) and torch.equal(ps1.cpu(), want[2]) and torch.equal(ps2.cpu(), want[3])
    assert torch.equal(c_map.cpu(), want[5].reshape(-1).clamp(min=-1))
    tiles = []
    for e in range(experts):
        first, end = int(want[0][e]), int(want[0][e + 1])
        tiles += [[e, r, end, 0] for r in range(first, end, tile)]
    plan = plan.cpu()
    assert int(plan[0]) == len(tiles)
    assert torch.equal(plan[4:4 + 4 * len(tiles)].view(-1, 4), torch.tensor(tiles, dtype=torch.int32).view(-1, 4))


@pytest.mark.parametrize("slots,experts,tile", [(2048, 7, 64), (2049, 7, 64), (3073, 256, 16), (3100, 257, 256), (5000, 1, 256), (32767, 256, 256), (32768, 31, 64)])
def test_several_segments(gpu, slots, experts, tile):
    """Both sides of the lines for several segments (2048 slots, 256 experts), short last segments, one expert with nearly all slots."""
    test_tables_and_plan(gpu, slots, experts, tile)


def test_limits_of_one_block(gpu):
    from sglang_amd import _lib

    lib = _lib.load()
    t = torch.zeros(64, dtype=torch.int32, device=gpu)
    p = t.data_ptr()
    assert lib.sglq_prepare_moe_layer(p, p, p, p, p, 32769, 4, 1, 1, 64, 8, p, None) == 2
    assert lib.sglq_prepare_moe_layer(p, p, p, p, p, 64, 513, 1, 1, 64, 8, p, None) == 2
    assert lib.sglq_prepare_moe_layer(p, p, p, p, p, 64, 4, 1, 1, 64, 8, None, None) == 1


@pytest.mark.parametrize("m,topk,e,n,k,dtype,weights", [(1, 1, 4, 128, 512, torch.bfloat16, torch.float32), (16, 8, 32, 256, 1024, torch.float16, torch.float32),
                                                        (333, 4, 9, 384, 256, torch.bfloat16, torch.bfloat16), (700, 6, 3, 512, 640, torch.bfloat16, torch.float32),
                                                        (11000, 3, 5, 128, 256, torch.bfloat16, torch.float32)])
def test_layer_host_path(gpu, monkeypatch, m, topk, e, n, k, dtype, weights):
    """One block's tables up to 32768 slots, the three-launch tables beyond; plans shared by the two GEMMs and not."""
    from sglang_amd import _lib
    from sglang_amd.moe import cutlass_moe

    _lib.load()
    print("layer", m, topk, e, n, k, dtype, weights, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m)
    rnd = lambda *s: torch.randn(s, generator=g, device=gpu)
    x = rnd(m, k).to(dtype)
    w1, w2 = rnd(e, 2 * n, k).to(torch.float8_e4m3fn).transpose(1, 2), rnd(e, k, n).to(torch.float8_e4m3fn).transpose(1, 2)
    s1 = (torch.rand((e, 2 * n // 128, k // 128), generator=g, device=gpu) * 1e-2 + 1e-3).transpose(1, 2)
    s2 = (torch.rand((e, k // 128, n // 128), generator=g, device=gpu) * 1e-2 + 1e-3).transpose(1, 2)
    tw, ids = torch.topk(torch.softmax(rnd(m, e), dim=-1), min(topk, e), dim=-1)
    ids = ids.to(torch.int32)
    if m > 8:
        ids[5, 0] = -1
    i64 = torch.empty((e,), dtype=torch.int64, device=gpu)
    tables = lambda: (torch.empty((e + 1,), dtype=torch.int32, device=gpu), torch.empty((e, 3), dtype=torch.int32, device=gpu), torch.empty((e, 3), dtype=torch.int32, device=gpu))
    ws = torch.empty((1 << 22,), dtype=torch.uint8, device=gpu)
    layer = lambda t: cutlass_moe.cutlass_fused_experts_fp8(x, w1, w2, s1, s2, tw.to(weights), ids, i64, i64, i64, i64, ws, i64, i64, i64, i64, i64, *t)
    got_t = tables()
    got = layer(got_t)
    assert _lib.native.experts(x, w1, w2, s1, s2, tw.to(weights), ids, *tables()) is not None

    class Off:
        experts = staticmethod(lambda *a: None)

    monkeypatch.setattr(cutlass_moe, "native", Off)
    want_t = tables()
    want = layer(want_t)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for a, b in zip(got_t, want_t):
        assert torch.equal(a, b)


# (in one launch: blocks of the gathered GEMM walk several tiles of three K blocks; beyond it: GEMM 2 takes the plan that GEMM 1 left, or forms its own)
@pytest.mark.parametrize("m,topk,e,n,k,one_launch,gathers,shared", [(4000, 8, 8, 768, 384, True, 1, True), (5000, 8, 6, 512, 640, False, 1, True),
                                                                    (12000, 3, 5, 256, 512, False, 1, False), (11000, 3, 5, 512, 256, False, 0, False)])
def test_layer_host_path_of_long_prompts(gpu, monkeypatch, m, topk, e, n, k, one_launch, gathers, shared):
    from sglang_amd import _lib

    lib, rows = _lib.load(), m * topk
    assert (rows <= 32768) == one_launch and topk > 2 and lib.sglq_grouped_gathers(e, rows, k) == gathers
    assert (lib.sglq_grouped_plan_rows(e, rows, k) == lib.sglq_grouped_plan_rows(e, rows, n)) == shared
    test_layer_host_path(gpu, monkeypatch, m, topk, e, n, k, torch.bfloat16, torch.float32)
