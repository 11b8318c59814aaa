"""The expert layer's first GEMM gathering its activation rows (sglq_fp8_blockwise_scaled_grouped_mm_gathered) against the same GEMM on
rows laid out expert by expert, bit for bit: ragged and empty experts, slots routed to nobody, the fewest K blocks, both plans."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,topk,e,n,k,dtype,empty", [(300, 2, 3, 128, 384, torch.bfloat16, False), (515, 3, 4, 192, 512, torch.float16, True),
                                                      (700, 6, 9, 384, 640, torch.bfloat16, True), (641, 1, 1, 128, 1152, torch.bfloat16, False),
                                                      (2500, 4, 5, 256, 1024, torch.bfloat16, False), (4099, 8, 8, 128, 384, torch.bfloat16, True)])
@pytest.mark.parametrize("planned", [True, False])
def test_gathered_rows(gpu, m, topk, e, n, k, dtype, empty, planned):
    from sglang_amd import _lib

    lib = _lib.load()
    rows = m * topk
    if planned and rows > 32768:
        pytest.skip("tables in one launch take up to 32768 slots")
    print("gathered", m, topk, e, n, k, dtype, empty, planned, flush=True)
    assert lib.sglq_grouped_gathers(e, rows, k) == 1
    g = torch.Generator(device="cuda").manual_seed(rows + e)
    x = torch.randn((m, k), generator=g, device=gpu).to(dtype)
    w = torch.randn((e, 2 * n, k), generator=g, device=gpu).to(torch.float8_e4m3fn)
    sw = torch.rand((e, 2 * n // 128, k // 128), generator=g, device=gpu) * 1e-2 + 1e-3
    ids = torch.topk(torch.rand((m, e), generator=g, device=gpu), topk, dim=1)[1].to(torch.int32).contiguous()
    if empty:
        ids[ids == e // 2] = e - 1  # an expert without rows, one with twice its share
        ids[::7, 0] = -1
    i32 = lambda *shape: torch.full(shape, 1 << 30, dtype=torch.int32, device=gpu)  # (tails of the row map name no token)
    offsets, ps1, ps2, slot_map, row_map = i32(e + 1), i32(e, 3), i32(e, 3), i32(rows), i32(rows)
    tiles = rows // 256 + e
    plan = i32(4 * (tiles + 1))
    st, code, out_code = _lib.stream_ptr(gpu), 0 if dtype == torch.bfloat16 else 1, 0 if dtype == torch.bfloat16 else 1
    p = lambda t: t.data_ptr()
    if planned:
        rc = lib.sglq_prepare_moe_layer_rows(p(ids), p(offsets), p(ps1), p(ps2), p(slot_map), p(row_map), topk, rows, e, n, k, 256, tiles, p(plan), st)
    else:
        slot_map.fill_(-1)
        rc = lib.sglq_prepare_moe_input(p(ids), p(offsets), None, p(ps1), p(ps2), p(row_map), p(slot_map), rows, topk, e, n, k, st)
    _lib.check(rc, "tables")
    routed = int(offsets[-1])
    live = slot_map >= 0
    assert torch.equal(row_map[slot_map[live].long()], (torch.arange(rows, device=gpu, dtype=torch.int32) // topk)[live])
    codes = lambda r: torch.zeros((r, k), dtype=torch.float8_e4m3fn, device=gpu)
    q, q_once = codes(rows), codes(m)
    s, s_once = torch.ones((k // 128, rows), device=gpu), torch.ones((k // 128, rows), device=gpu)
    _lib.check(lib.sglq_per_token_group_quant_fp8_scatter_cm(p(x), code, p(q), p(s), p(slot_map), m, k, topk, rows, 1e-10, st), "scatter")
    _lib.check(lib.sglq_per_token_group_quant_fp8_scatter_scales_cm(p(x), code, p(q_once), p(s_once), p(slot_map), m, k, topk, rows, 1e-10, st), "scales")
    assert torch.equal(s, s_once)
    assert torch.equal(q_once.view(torch.uint8)[row_map[:routed].long()], q.view(torch.uint8)[:routed])
    y, z = (torch.full((rows, 2 * n), 3.0, dtype=dtype, device=gpu) for _ in range(2))
    tail = lambda s: (p(w), k, 2 * n * k, p(s), 1, rows, p(sw), sw.stride(0), sw.stride(2), sw.stride(1))
    if planned:
        rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_planned(p(q), k, *tail(s), p(y), 2 * n, out_code, 256, e, rows, 2 * n, k, p(plan), plan.numel() * 4, st)
    else:
        rc = lib.sglq_fp8_blockwise_scaled_grouped_mm(p(q), k, *tail(s), p(y), 2 * n, out_code, p(ps1), p(offsets), e, rows, 2 * n, k, p(plan),
                                                      plan.numel() * 4, st)
    _lib.check(rc, "grouped")
    rc = lib.sglq_fp8_blockwise_scaled_grouped_mm_gathered(p(q_once), k, m, p(row_map), *tail(s_once), p(z), 2 * n, out_code, p(ps1), p(offsets),
                                                           256 if planned else 0, e, rows, 2 * n, k, p(plan), plan.numel() * 4, st)
    _lib.check(rc, "gathered")
    assert torch.isfinite(z.float()).all() and bool((z[:routed] != 3.0).any())
    assert torch.equal(y, z)


# Blocks that walk three to five tiles each: the next tiles' row maps, K blocks of theirs read in the steps before, stores left in flight, tiles of
# other heights behind each other (150 rows an expert) and columns that end inside a tile; three K blocks leave no step between the first and the last but one.
@pytest.mark.parametrize("m,topk,e,n,dtype,empty", [(4000, 8, 8, 768, torch.bfloat16, False), (4001, 8, 9, 1088, torch.float16, True), (3000, 4, 80, 1152, torch.bfloat16, True)])
@pytest.mark.parametrize("k", [384, 512, 640, 1024])
@pytest.mark.parametrize("planned", [True, False])
def test_gathered_blocks_walk_several_tiles(gpu, m, topk, e, n, k, dtype, empty, planned):
    assert max(m * topk // 256, e - 1) * (2 * n // 256) > 2 * torch.cuda.get_device_properties(gpu).multi_processor_count
    test_gathered_rows(gpu, m, topk, e, n, k, dtype, empty, planned)


def test_sizes_that_do_not_gather(gpu):
    from sglang_amd import _lib

    lib = _lib.load()
    t = torch.zeros(4096, dtype=torch.int32, device=gpu)
    p = t.data_ptr()
    assert lib.sglq_grouped_gathers(4, 64, 1024) == 0 and lib.sglq_grouped_gathers(4, 4096, 256) == 0
    call = lambda row_map, total, K: lib.sglq_fp8_blockwise_scaled_grouped_mm_gathered(p, K, 4, row_map, p, K, 256 * K, p, 1, total, p, 1, 1, 1, p, 256, 0, p, p,
                                                                                     0, 1, total, 256, K, p, 16384, None)
    assert call(p, 8, 512) == 1 and call(None, 1024, 512) == 1
