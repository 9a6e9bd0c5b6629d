"""NaN among the inputs of the fp32 kernels of the single representation: it reaches what depends on it and nothing else."""
import pytest
import torch

from gpu_util import lib  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair
import of3pair.functional

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _attention(n, seed):
    gen = torch.Generator().manual_seed(seed)
    p = orc.make_attention_pair_bias_params(gen, 384, 32, 24, 16)
    a, z = torch.randn(1, n, 384, generator=gen), orc.make_pair_input(seed + 1, (1,), n, 32)
    mod = of3pair.AttentionPairBias(384, 384, 384, 384, 32, 24, 16)
    mod.load_state_dict(p, strict=True)
    return a, z, p, mod.to(DEV).eval()


@pytest.mark.parametrize("n", [7, 33, 129, 200])
def test_nan_logit_is_no_masked_key(n):
    """One element of z is NaN: the query whose pair bias it feeds is NaN, as softmax gives it, the others are finite."""
    lib()
    a, z, p, mod = _attention(n, 6100 + n)
    for query, key in ((0, n - 1), (n // 2, 0), (n - 1, n // 2)):
        z[0, query, key, 5] = float("nan")
        want = orc.attention_pair_bias(a, z, None, p, 16)
        got = mod(a.to(DEV), z.to(DEV)).cpu()
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.isnan(got[0, query]).all()
    mask = torch.ones(1, n)
    mask[0, n // 3] = float("nan")
    assert torch.isnan(mod(a.to(DEV), z.to(DEV), mask=mask.to(DEV))).all()


@pytest.mark.parametrize("n,open_keys", [(70, slice(32, 70)), (70, slice(5, 6)), (200, slice(199, 200)), (300, slice(130, 140)), (40, slice(0, 0))])
def test_keys_at_minus_infinity(n, open_keys):
    """A pair bias of -inf leaves a key out, also where that leaves a whole tile of a query without any (and NaN where
    it leaves the query without any)."""
    lib()
    a, _, p, mod = _attention(n, 6200 + n)
    bias = torch.randn(1, 16, n, n, generator=torch.Generator().manual_seed(6300 + n))
    closed = torch.ones(n, dtype=torch.bool)
    closed[open_keys] = False
    for query in (0, n // 2, n - 1):
        bias[0, :, query, closed] = float("-inf")
    m = mod.mha
    got = of3pair.functional.attention_pair_bias(
        a.to(DEV), None, None, mod.layer_norm_a.weight, mod.layer_norm_a.bias, None, None, None, m.linear_q.weight, m.linear_q.bias,
        m.linear_k.weight, m.linear_v.weight, m.linear_g.weight, m.linear_o.weight, no_heads=16, _bias=bias.to(DEV)).cpu()
    q = {k: v.double() for k, v in p.items()}
    an = torch.nn.functional.layer_norm(a.double(), (384,), q["layer_norm_a.weight"], q["layer_norm_a.bias"])

    def heads(x):
        return x.view(1, n, 16, 24).transpose(1, 2)

    query = heads(an @ q["mha.linear_q.weight"].T + q["mha.linear_q.bias"]) / 24 ** 0.5
    key, value = heads(an @ q["mha.linear_k.weight"].T), heads(an @ q["mha.linear_v.weight"].T)
    o = (query @ key.transpose(-1, -2) + bias.double()).softmax(-1) @ value
    want = (o.transpose(1, 2).reshape(1, n, 384) * torch.sigmoid(an @ q["mha.linear_g.weight"].T)) @ q["mha.linear_o.weight"].T
    assert torch.equal(got.isnan(), want.isnan())
    scale = max(1.0, float(want.nan_to_num().abs().max()))
    # the bound of the tile tests: 384-term fp32 sums, four of them in a row
    assert float((got.double() - want).nan_to_num().abs().max()) <= 5e-6 * scale
