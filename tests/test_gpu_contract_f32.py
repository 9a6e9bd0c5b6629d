"""Both tiles of the fp32 contraction (contract_x3_launch) on either side of the rule, at lengths that fill their tiles, leave one
column or one 32 x 32 part of them, and leave waves without any.  Tolerance: as in the tests of the passes around it."""
import pytest

import test_gpu_pass_f32 as passes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch,c", [(64, 1, 128), (65, 2, 128), (97, 1, 64), (192, 1, 128), (129, 1, 128), (193, 3, 64), (225, 1, 128),
                                       (256, 2, 128), (257, 1, 128), (320, 1, 64), (321, 1, 128), (353, 1, 128)])
def test_trimul(n, batch, c):
    passes.test_trimul(n, batch, c)
