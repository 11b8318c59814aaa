"""Which kernel takes 65 to 128 rows of wide weights, on both sides of the line between the pipelined 128-row kernel and the ring: named, and compared with the generic kernel."""
import pytest
from test_gemm_selection_gpu import test_power_of_two_scales_up_to_128_rows as power_of_two_scales, test_the_rules_choose as the_rules_choose

pytestmark = pytest.mark.gpu
RING, PIPE_128 = "gemm_ring_kernel", "gemm_pipe_kernel<128 rows>+splitk_reduce_kernel"


# (more than 16384 weight rows; long K on few tiles; fewer weight rows; columns that end inside a tile)
@pytest.mark.parametrize("kind,m,n,k,kernel", [("fp8", 128, 17408, 5120, RING), ("block", 65, 20480, 5120, RING), ("i8", 100, 23312, 4480, RING), ("block_i8", 120, 17408, 5120, RING),
                                               ("fp8", 128, 16896, 14208, PIPE_128), ("i8", 80, 13824, 5120, "gemm_kwave_kernel"), ("i8", 66, 18432, 7168, RING)])
def test_wide_weights(gpu, kind, m, n, k, kernel):
    the_rules_choose(gpu, kind, m, n, k, kernel)


@pytest.mark.parametrize("m,n,k,kernel,packed_kernel", [(72, 20480, 5120, RING, RING), (128, 18432, 7168, RING, RING)])
def test_wide_weights_of_power_of_two_scales(gpu, m, n, k, kernel, packed_kernel):
    power_of_two_scales(gpu, m, n, k, kernel, packed_kernel)
