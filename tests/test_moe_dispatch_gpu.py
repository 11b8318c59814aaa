"""Which kernels an expert layer launches, by its sizes: the host path's choices (row tiles, walks, rows gathered, the quantization beside the tables, the activation behind GEMM 1), in order.
What they compute is compared in the other test_moe files."""
import re

import pytest
import torch
from helpers import launches

pytestmark = pytest.mark.gpu

TABLES, TABLES_QUANT, QUANT = "moe_tables_kernelILin1E", "moe_tables_kernelILi[01]E", "group_quant_scatter_kernel"
FEW_32, FEW_64 = "gemm_few_rows_kernelILi[01]ELi32E", "gemm_few_rows_kernelILi[01]ELi64E"
ROWS_32, RING, PIPE_128 = "gemm_kernelILi0ELi32E", "gemm_ring_kernel", "gemm_pipe_kernelILi0ELi[01]ELi3ELi128E"
GATHERED, WALKED, WALKED_GATHERED, ACTIVATES, ACTIVATES_GATHERED = (f"gemm_pipe_kernelILi0ELi[01]ELi{mode}ELi256E" for mode in (5, 6, 7, 8, 9))
SILU, SUM = "silu_mul_group_quant_kernel", "shuffle_mul_sum_kernel"


# (few rows with the activation and, of too few K blocks, without it; 64 rows; above 2048 slots and 512 tokens the quantization by itself; 32 rows from 12 rows an expert on; no 32 rows on long K;
# the rows of fewer and more than 129 rows an expert, of one or two experts a token and of more; other heights; an intermediate size without walks)
@pytest.mark.parametrize("m,topk,e,n,k,kernels", [
    (16, 4, 16, 1536, 1536, [TABLES_QUANT, FEW_32, ROWS_32, SUM]),
    (16, 4, 16, 1536, 1408, [TABLES_QUANT, ROWS_32, SILU, ROWS_32, SUM]),
    (122, 4, 16, 1536, 1536, [TABLES_QUANT, FEW_64, RING, SUM]),
    (90, 4, 16, 1024, 2048, [TABLES_QUANT, RING, SILU, RING, SUM]),
    (480, 4, 60, 1408, 1536, [TABLES_QUANT, FEW_32, ROWS_32, SUM]),
    (121, 3, 24, 384, 1152, [TABLES_QUANT, FEW_32, ROWS_32, SUM]),
    (1046, 1, 66, 512, 1280, [TABLES, QUANT, ROWS_32, SILU, ROWS_32, SUM]),
    (300, 8, 64, 768, 2048, [TABLES, QUANT, FEW_32, ROWS_32, SUM]),
    (79, 3, 13, 1024, 7168, [TABLES_QUANT, RING, SILU, RING, SUM]),
    (300, 8, 32, 1024, 1024, [TABLES, QUANT, ACTIVATES_GATHERED, WALKED, SUM]),
    (900, 6, 6, 384, 512, [TABLES, QUANT, WALKED_GATHERED, SILU, WALKED, SUM]),
    (1400, 6, 6, 384, 512, [TABLES, QUANT, ACTIVATES_GATHERED, WALKED, SUM]),
    (1400, 2, 5, 384, 1024, [TABLES, QUANT, WALKED, SILU, WALKED, SUM]),
    (600, 2, 5, 2048, 1024, [TABLES, QUANT, PIPE_128, SILU, PIPE_128, SUM]),
    (1326, 1, 9, 384, 2048, [TABLES, QUANT, RING, SILU, RING, SUM]),
    (900, 6, 6, 256, 512, [TABLES, QUANT, GATHERED, SILU, "grouped_plan_kernel", "gemm_kernelILi0ELi128E", SUM]),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_launches(gpu, m, topk, e, n, k, kernels, dtype):
    from sglang_amd._lib import load, native

    print("launches", m, topk, e, n, k, dtype, flush=True)
    load()
    fp8 = lambda *s: torch.zeros(s, dtype=torch.uint8, device=gpu).view(torch.float8_e4m3fn).transpose(1, 2)
    scales = lambda *s: torch.ones(s, device=gpu).transpose(1, 2)
    i32 = lambda *s: torch.zeros(s, dtype=torch.int32, device=gpu)
    args = (torch.zeros((m, k), dtype=dtype, device=gpu), fp8(e, 2 * n, k), fp8(e, k, n), scales(e, 2 * n // 128, k // 128), scales(e, k // 128, n // 128),
            torch.ones((m, topk), device=gpu), torch.arange(m * topk, dtype=torch.int32, device=gpu).view(m, topk) % e, i32(e + 1), i32(e, 3), i32(e, 3))
    assert native.experts(*args) is not None
    names = launches(lambda: native.experts(*args))
    assert len(names) == len(kernels) and all(re.search(want, name) for want, name in zip(kernels, names)), names
