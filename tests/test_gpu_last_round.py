"""bf16 position-wise passes whose last round of tiles is dealt in pieces (last_round in openfold-3_amd/csrc/of3_tiles.h): halves
and quarters of a tile, as the only round or after whole ones, rows that end inside a piece, two-piece ragged columns."""
import pytest

import test_gpu_stages as stages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,d,n,batch", [(128, 32, 96, 1), (128, 32, 110, 1), (128, 32, 170, 1), (128, 32, 187, 1), (128, 32, 200, 1),
                                         (128, 32, 256, 1), (128, 32, 81, 2), (64, 16, 91, 1), (64, 16, 187, 2), (64, 16, 200, 1)])
def test_stages(c, d, n, batch):
    for flag in (False, True):
        stages.test_trimul_proj(flag, c, n, batch)
        stages.test_trimul_out(int(flag), c, n, batch)
        stages.test_triattn_proj(flag, c, d, n, batch)
        stages.test_triattn_out(flag, int(flag), c, d, n, batch)
