"""The shapes that the fused quantize-and-multiply kernels take for the launch they save: short K up to 8 rows."""
import pytest

import test_fused_linear_gpu as block
import test_fused_token_linear_gpu as token

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mnk,fused", [((1, 1024, 512), True), ((4, 2048, 4096), True), ((4, 1016, 1024), False), ((5, 4096, 4096), True),
                                       ((8, 4104, 1024), True), ((8, 4104, 1152), False), ((8, 1024, 4224), False)])
def test_block_fp8_linear_short_k(gpu, mnk, fused):
    block.check_case(gpu, *mnk, seed=sum(mnk), with_bias=True, outliers=True, expect_fused=fused)


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("mnk,fused", [((3, 1024, 2560), True), ((8, 4096, 1024), True), ((8, 2048, 1152), False), ((4, 4104, 1024), False)])
def test_token_linear_short_k(gpu, kind, mnk, fused):
    token.check_case(gpu, kind, *mnk, seed=sum(mnk), with_bias=True, outliers=True, expect_fused=fused)
