"""The forms of the triangle attention core (triattn_flash_launch) that the smaller stage tests do not reach: 128 queries of two
waves per row (heads of 32, long launches) and of one wave per row (heads of 16, long launches), at ragged lengths, with
masked rows and runs, and with logits that need the second pass; lengths on either side of the rule."""
import pytest

import test_gpu_stages as stages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,n,B,logit_scale", [(32, 449, 1, 1.0), (32, 418, 1, 40.0), (32, 384, 1, 1.0), (32, 416, 1, 1.0),
                                               (16, 247, 9, 1.0), (16, 256, 7, 40.0), (16, 225, 9, 1.0), (16, 384, 2, 1.0)])
def test_forms(D, n, B, logit_scale):
    stages.test_triattn_flash(D, n, B, logit_scale)


@pytest.mark.parametrize("D,n,B,pads", [(32, 470, 1, "tail"), (32, 450, 1, "outer"), (16, 250, 8, "tail"), (16, 240, 8, "head")])
def test_padding(D, n, B, pads):
    stages.test_triattn_flash_padding_masks(D, n, B, pads)
