"""Rows whose keys are all masked: where every row of a work-group is such a row the attention core looks whether all logits are level
(the mask bias takes up what the bias and q k add) and takes the mean of v; beside other rows, or with logits too large for that,
it goes through the softmax with running maxima.  The rows of an attention do not depend on one another's masks, so both give the
same bits."""
import pytest
import torch

from gpu_util import lib  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("c,d", [(64, 16), (128, 32)])
@pytest.mark.parametrize("n", [9, 33, 64, 150, 451])  # one key tile that is not full, odd and even numbers of them, every form of the core
@pytest.mark.parametrize("what", ["ordinary", "large bias", "large logit", "nan"])
def test_level_rows(what, n, c, d, dtype):
    lib()
    gen = torch.Generator().manual_seed(8700 + n + c)
    p = orc.make_triattn_params(gen, c, d, c // d)
    name = [k for k in p if p[k].dim() == 2 and p[k].shape[0] == c // d][0]
    z = orc.make_pair_input(8701, (1,), n, c)
    if what == "large bias":
        p[name] = p[name] * 100.0
    elif what == "large logit":  # one of a masked row's, its last query and key
        z[0, 5, n - 1] = z[0, 5, n - 1] * 0 + torch.linspace(-1, 1, c)
        q = [k for k in p if k.endswith("linear_q.weight")][0]
        p[q] = p[q] * 300.0
    elif what == "nan":
        z[0, 5, n - 1, 3] = float("nan")
    m = of3pair.TriangleAttention(c, d, c // d)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).to(dtype).eval()
    print("level rows", what, n, c, dtype, flush=True)
    out = []
    for rows in (range(4, 8), (5,)):  # whole groups of rows that share a work-group, and one row of a group
        mask = torch.ones(1, n, n)
        mask[:, list(rows)] = 0.0
        out.append(m(z.to(DEV).to(dtype), mask.to(DEV))[0, 5].cpu())
    assert out[0].shape == (n, c)
    assert torch.equal(torch.isnan(out[0]), torch.isnan(out[1]))
    assert torch.equal(torch.nan_to_num(out[0].float()), torch.nan_to_num(out[1].float()))
    assert bool(torch.isnan(out[0]).any()) == (what == "nan")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("c,d", [(64, 16), (128, 32)])
# keys on both sides of the tiles after which the core looks: 2, 8 of 32 keys, the last
@pytest.mark.parametrize("n,key", [(65, 0), (65, 40), (65, 64), (451, 31), (451, 63), (451, 64), (451, 250), (451, 256), (451, 450)])
def test_one_logit_is_not_level(n, key, c, d, dtype):
    """The triangle bias of one query and key alone is too large for the mask bias to take up."""
    lib()
    gen = torch.Generator().manual_seed(8720 + c)
    p = orc.make_triattn_params(gen, c, d, c // d)
    name = [k for k in p if p[k].dim() == 2 and p[k].shape[0] == c // d][0]
    p[name][:, 0] = 100.0
    p["layer_norm.bias"][0] = 0.0
    z = orc.make_pair_input(8721, (1,), n, c)
    z = z - z.mean(-1, keepdim=True)
    z[..., 0] = 0.0
    query = n - 2
    z[0, query, key, 0] = 1e3
    m = of3pair.TriangleAttention(c, d, c // d)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).to(dtype).eval()
    print("one logit", key, n, c, dtype, flush=True)
    out = []
    for rows in (range(4, 8), (5,)):
        mask = torch.ones(1, n, n)
        mask[:, list(rows)] = 0.0
        out.append(m(z.to(DEV).to(dtype), mask.to(DEV))[0, 5].cpu())
    assert torch.equal(out[0], out[1]) and bool(torch.isfinite(out[0]).all())
