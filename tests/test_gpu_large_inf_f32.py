"""fp32 triangle attention with other mask biases than -1e9: near fp32's largest numbers, where they are multiplied with the scales of q
and k (two fp16 terms: 64 and 128 channels), and with odd mantissas, to which the matrix instructions do not add a small logit as it
should be (all biases but 1e9 here; 96 channels: three bf16 terms, 40: no matrix instructions)."""
import pytest
import torch

from gpu_util import lib, report  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("c,d", [(64, 16), (128, 32), (96, 32), (40, 8)])
@pytest.mark.parametrize("size", [1e-3, 1.0])  # of the weights: the smaller they are the larger the scales
@pytest.mark.parametrize("inf", [1e9, 1e10, 1e15, 1e25, 1e33, 1e38])
def test_large_inf(inf, size, c, d):
    lib()
    n = 45
    gen = torch.Generator().manual_seed(9000 + c)
    p = orc.make_triattn_params(gen, c, d, c // d)
    for name in ("mha.linear_q.weight", "mha.linear_k.weight"):
        p[name] = p[name] * size
    z = orc.make_pair_input(9001, (1,), n, c)
    mask = (torch.rand(1, n, n, generator=gen) > 0.2).float()
    mask[:, 4:8] = 0.0  # rows of masked keys: the mean of v
    mask[:, 20] = 0.0
    mask[:, 30, ::2] = 0.0
    mask[:, 30, 1::2] = 0.5  # a row whose largest mask value is below 1
    print("large inf", inf, size, c, d, flush=True)
    # at 1e9 fp32 takes up the logits of a row of masked keys, 64 bits do not
    p64 = {k: v.double() for k, v in p.items()}
    want = orc.triattn_update(z.double(), mask.double(), p64, c // d, inf=max(inf, 1e25))
    m = of3pair.TriangleAttention(c, d, c // d, inf=inf)
    m.load_state_dict(p, strict=True)
    got = m.to(DEV).eval()(z.to(DEV), mask.to(DEV)).cpu()
    # 1e-5 of the largest value as in the other fp32 tests of the module; at 5e8 (row 30) fp32 takes up logits of 16 and less
    rows = list(range(n))
    report("update", got[:, rows], want[:, rows], atol=1e-5 * float(want.abs().max()))
    assert got.isfinite().all()
