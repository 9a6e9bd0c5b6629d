"""The forms of the triangle attention core (triattn_flash_launch) that the smaller stage tests do not reach: 128 queries of two
waves per row (heads of 32) and of one wave per row (heads of 16), and 96 of one wave per row, whose last range holds one, two or three
32-query tiles, at ragged lengths, with masked rows and runs, and with logits that need the second pass; lengths on either side of the rule."""
import pytest

import test_gpu_fp32 as fp32
import test_gpu_stages as stages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,n,B,logit_scale", [(32, 449, 1, 1.0), (32, 418, 1, 40.0), (32, 384, 1, 1.0), (32, 416, 1, 1.0),
                                               (32, 200, 2, 1.0), (32, 500, 1, 40.0), (32, 259, 1, 1.0), (32, 343, 1, 40.0),
                                               (32, 130, 2, 40.0), (16, 187, 2, 40.0), (16, 130, 3, 1.0), (16, 390, 1, 40.0), (32, 390, 3, 1.0),
                                               (16, 247, 9, 1.0), (16, 256, 7, 40.0), (16, 225, 9, 1.0), (16, 384, 2, 1.0)])
def test_forms(D, n, B, logit_scale):
    stages.test_triattn_flash(D, n, B, logit_scale)


@pytest.mark.parametrize("D,n,B,pads", [(32, 470, 1, "tail"), (32, 450, 1, "outer"), (32, 500, 1, "tail"), (32, 360, 1, "head"),
                                        (16, 187, 2, "tail"), (16, 288, 2, "middle"), (16, 250, 8, "tail"), (16, 240, 8, "head")])
def test_padding(D, n, B, pads):
    stages.test_triattn_flash_padding_masks(D, n, B, pads)


# fp32: work-groups of 64 queries (a last range of 128 that is at most half full; heads of 32, one round of launches: a quarter) and of 128, with masked rows and columns
@pytest.mark.parametrize("c,d,n,batch", [(128, 32, 129, ()), (128, 32, 160, ()), (128, 32, 161, ()), (128, 32, 161, (2,)), (128, 32, 193, ()),
                                         (128, 32, 290, ()), (64, 16, 129, (2,)), (64, 16, 192, ()), (64, 16, 193, ())])
def test_fp32_forms(c, d, n, batch):
    fp32.test_triattn_fp32(True, c, d, 4, n, batch, True)
