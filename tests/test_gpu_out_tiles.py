"""bf16 output passes on tiles of 64 positions (out_tile_positions in openfold-3_amd/csrc/of3_tiles.h) and at the edges of their rule: rows that are
whole multiples of 64 but not of 128, ragged columns of one and of two pieces, last rounds in halves of a tile, and 897 tokens, where
the planes of x are 1024 wide and the pass that reads them goes on in tiles of 128.  Above three rounds (331 and 320 tokens, two
tensors of 64 channels) there are no pieces, and rows leave whole."""
import pytest

import test_gpu_stages as stages


@pytest.mark.gpu
@pytest.mark.parametrize("c,d,n,batch", [(128, 32, 192, 1), (128, 32, 225, 1), (128, 32, 257, 1), (128, 32, 321, 1), (128, 32, 48, 9), (64, 16, 192, 1),
                                         (64, 16, 193, 2), (64, 16, 250, 1), (64, 16, 320, 2), (64, 16, 331, 2), (64, 16, 384, 2), (128, 32, 512, 1), (128, 32, 896, 1), (128, 32, 897, 1)])
def test_stages(c, d, n, batch):
    stages.test_trimul_out(1, c, n, batch)
    for starting in (False, True):
        stages.test_triattn_out(starting, 1, c, d, n, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("transposed", [False, True])
def test_attention_long_rows(transposed):
    """Above 1536 tokens the attention's pass takes tiles of 128: here off their multiples, so that a tile lies in two rows."""
    stages.test_triattn_out(transposed, 1, 128, 32, 1537, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [897, 1024])
def test_planes_of_1024(n):
    """64 channels: the planes of x are 1024 wide and the pass that reads them takes tiles of 128, ragged rows and whole ones."""
    stages.test_trimul_out(1, 64, n, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(256, 1), (257, 1), (187, 2), (200, 2), (331, 1), (63, 9)])
def test_input_pass_64(n, batch):
    """64 channels on both sides of two tiles per CU (256 CUs: 512 tiles at 256 tokens, 585 at 257), where work-groups of four waves take over from
    those of eight, with pieces of both sizes in the last round and without."""
    for incoming in (False, True):
        stages.test_trimul_proj(incoming, 64, n, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(230, 1), (257, 1), (384, 1), (300, 2), (256, 4), (512, 2), (513, 2), (500, 3)])
def test_attention_input_pass_64(n, batch):
    """Two work-groups to a CU from one tile of 128 positions per CU (256 CUs) up to sixteen (512 tokens, two tensors: 4096 tiles; 513: more), with pieces in the
    last round and without, whole rows and ragged ones."""
    for ending in (False, True):
        stages.test_triattn_proj(ending, 64, 16, n, batch)
