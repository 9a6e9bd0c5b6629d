"""bf16 output passes on tiles of 64 positions (out_tile_positions in openfold-3_amd/csrc/of3_tiles.h) and at the edges of their rule: rows that are
whole multiples of 64 but not of 128, ragged columns of one and of two pieces, last rounds in halves of a tile, and 897 tokens, where
the planes of x are 1024 wide and the pass that reads them goes on in tiles of 128."""
import pytest

import test_gpu_stages as stages


@pytest.mark.gpu
@pytest.mark.parametrize("c,d,n,batch", [(128, 32, 192, 1), (128, 32, 225, 1), (128, 32, 257, 1), (128, 32, 321, 1), (128, 32, 48, 9), (64, 16, 192, 1),
                                         (64, 16, 193, 2), (64, 16, 250, 1), (128, 32, 896, 1), (128, 32, 897, 1)])
def test_stages(c, d, n, batch):
    stages.test_trimul_out(1, c, n, batch)
    for starting in (False, True):
        stages.test_triattn_out(starting, 1, c, d, n, batch)
