"""Both tiles of the fp32 output products over s (small_tiles) on either side of the rule, at ragged row counts; the tiles of 16 at their edges."""
import pytest

import test_gpu_single_x3 as single

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,c,n_mult,masked", [(15, 64, 1, True), (17, 384, 4, False), (336, 384, 2, True), (337, 384, 2, True), (257, 512, 4, False)])
def test_row_transition(rows, c, n_mult, masked):
    single.test_row_transition_fp32_tiles(rows, c, n_mult, masked)


@pytest.mark.parametrize("n,c_s,c_head,heads,mask", [(16, 64, 16, 2, None), (17, 384, 24, 16, "tail"), (335, 384, 24, 16, "tail"), (339, 384, 24, 16, None),
                                                     (260, 512, 32, 16, "tail")])
def test_attention_pair_bias(n, c_s, c_head, heads, mask):
    single.test_attention_pair_bias_fp32_tiles(n, c_s, c_head, heads, mask)
