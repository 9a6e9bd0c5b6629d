"""The bf16 contraction's tiles of 64 x 64 (contract_short_kernel): one to eight panels (fewer than its ring holds, as many, more), tiles that
are full, hold one 32 x 32 part in use, or leave waves without any.  The transposed form: test_gpu_pair_join.py, against this one."""
import pytest

import test_gpu_stages as stages

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [2, 3])
@pytest.mark.parametrize("n", [1, 33, 64, 65, 97, 128, 161, 192, 193, 225, 256])
def test_short(variant, n):
    stages.test_contract_ragged_n(variant, n)
