"""The fp32 attention input pass with two work-groups to a tile: as many tiles as half of the CUs, one more, a batch, ragged panels; heads of 16
and 32.  Tolerance: as in the tests of the passes around it."""
import pytest

import test_gpu_pass_f32 as passes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [16, 32])
@pytest.mark.parametrize("n,batch", [(64, 1), (43, 1), (32, 4), (65, 1), (7, 5)])
def test_triattn(n, batch, d):
    passes.test_triattn(n, batch, 128, d)
