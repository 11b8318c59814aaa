"""Which row tiles an expert layer's sizes choose on 256 CUs where K is long: 32-row tiles lose there below half a round and, from 1.9 rounds on, to three rounds of the ring's 64-row tiles."""
import pytest


# (0: the ring by rows alone.  Below half a round and from there; K of 33 blocks, where the line lies; three rounds of the ring and more; short K on both sides)
@pytest.mark.parametrize("m,topk,e,n,k,rows", [(79, 3, 13, 1024, 7168, 0), (115, 3, 20, 768, 5760, 0), (64, 4, 16, 1536, 5120, 32), (49, 7, 17, 768, 4224, 32), (49, 7, 17, 768, 4352, 0),
                                               (561, 7, 105, 384, 4480, 0), (143, 8, 30, 1408, 5632, 0), (559, 2, 31, 1280, 6400, 0), (858, 6, 160, 384, 5120, 32), (565, 4, 93, 640, 4480, 32),
                                               (143, 8, 30, 1408, 4224, 32), (44, 7, 22, 384, 2688, 32)])
def test_rows_of_a_layer(m, topk, e, n, k, rows):
    import torch

    from sglang_amd import _lib

    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are in rounds of 256 CUs")
    assert _lib.load().sglq_grouped_layer_rows(e, m, topk, n, k) == rows
