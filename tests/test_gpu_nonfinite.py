"""NaN, infinities and values above the largest bf16 in the fp32 kernels that split their operands into bf16 terms: they
reach what depends on them as in plain arithmetic, and nothing else."""
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


def _same(got, want, rtol=5e-5):
    """got (fp32) against want (64 bits, an infinity from the largest fp32 value on): NaN and infinities at the same
    places, the rest to rtol: sums of up to 160 terms of which one may be 1e38 times the others."""
    want = want.float()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[want.isinf()], want[want.isinf()])
    fin = want.isfinite()
    assert torch.allclose(got[fin], want[fin], rtol=rtol, atol=1e-5)


INF, HUGE = float("inf"), 3.4e38  # HUGE: above the largest bf16, 3.3895e38


@pytest.mark.parametrize("n,name,value", [(33, "wg", INF), (33, "wg", -HUGE), (33, "wo", -INF), (70, "wo", HUGE), (1, "wv", INF), (1, "wv", HUGE),
                                          (33, "wq", INF), (33, "key", 1e38), (161, "key", 1e38)])
def test_attention_keeps_infinities(n, name, value):
    """An infinite or very large weight: infinities, zeros of the gate and left-out keys as plain arithmetic gives them."""
    lib()
    c, gen = 32, torch.Generator().manual_seed(6400 + n)
    w = {k: torch.randn(c, c, generator=gen) / c ** 0.5 for k in ("wq", "wk", "wv", "wg", "wo")}
    bq = torch.zeros(c)
    a = torch.randn(1, n, c, generator=gen)
    if name == "key":
        # the first channel of key n / 2 is -inf, of every other one 0; that of every query is positive
        signs = torch.tensor([1.0, -1.0, 1.0, -1.0]).repeat(c // 4)
        a = signs.repeat(1, n, 1) * torch.tensor([1.0, -1.0])[torch.randint(2, (1, n, 1), generator=gen)]
        a[0, n // 2, :8] = torch.tensor([1.0, 1.0, 1.0, 1.0, -1.0, -1.0, -1.0, -1.0])
        w["wk"][0] = 0.0
        w["wk"][0, :4] = -value
        w["wq"][0] = 0.0
        bq[0] = 3.0
    else:
        w[name][2, 3] = value
    one, zero = torch.ones(c), torch.zeros(c)
    bias = torch.randn(1, 1, n, n, generator=gen)
    args = [t.to(DEV) for t in (one, zero)] + [None, None, None] + [t.to(DEV) for t in (w["wq"], bq, w["wk"], w["wv"], w["wg"], w["wo"])]
    got = of3pair.functional.attention_pair_bias(a.to(DEV), None, None, *args, no_heads=1, _bias=bias.to(DEV)).cpu()
    d = {k: v.double() for k, v in w.items()}
    an = torch.nn.functional.layer_norm(a.double(), (c,))
    if name == "key":  # what the logits come to (the zeros of the other keys are exact in 32 bits, not in 64)
        d["wk"][0] = 0.0
        bias[..., n // 2] = -INF
    q, k, v, g = an @ d["wq"].T + bq.double(), an @ d["wk"].T, an @ d["wv"].T, torch.sigmoid(an @ d["wg"].T)
    o = ((q @ k.transpose(-1, -2) / c ** 0.5 + bias[:, 0].double()).softmax(-1) @ v) * g
    if n == 1:
        o = o.float().double()  # what is stored between the kernels is fp32
    _same(got, o @ d["wo"].T)


@pytest.mark.parametrize("name,value", [("wa", INF), ("wa", HUGE), ("wb", INF), ("wb", -HUGE), ("wo", -INF), ("wo", HUGE)])
def test_row_transition_keeps_infinities(name, value):
    lib()
    c, hid, gen = 64, 128, torch.Generator().manual_seed(6500)
    w = {k: torch.randn(*s, generator=gen) / s[1] ** 0.5 for k, s in (("wa", (hid, c)), ("wb", (hid, c)), ("wo", (c, hid)))}
    w[name][5, 9] = value
    x = torch.randn(45, c, generator=gen)
    got = of3pair.functional.swiglu_transition(x.to(DEV), None, torch.ones(c, device=DEV), torch.zeros(c, device=DEV),
                                               *[w[k].to(DEV) for k in ("wa", "wb", "wo")]).cpu()
    d = {k: v.double() for k, v in w.items()}
    xn = torch.nn.functional.layer_norm(x.double(), (c,))
    ha, hb = (xn @ d["wa"].T).float(), (xn @ d["wb"].T).float()
    h = (ha * torch.sigmoid(ha)) * hb
    # a large hidden channel 5 is the whole sum, to the relative error of its two factors: sums of 64 terms that add up to
    # 8 in size, 64 * 2^-24 * 8 / 16 = 2e-6 absolute
    _same(got, h.double() @ d["wo"].T, rtol=5e-5 + 2e-6 / float(ha[:, 5].abs().min()) + 2e-6 / float(hb[:, 5].abs().min()))


@pytest.mark.parametrize("where,value,apply_ln", [("t", INF, False), ("t", HUGE, False), ("t", -INF, False), ("w", INF, True), ("w", -HUGE, True),
                                                  ("w", INF, False)])
def test_template_tail_keeps_infinities(where, value, apply_ln):
    lib()
    gen = torch.Generator().manual_seed(6600)
    t, w = torch.randn(2, 3, 7, 7, 64, generator=gen), torch.randn(128, 64, generator=gen)
    lw, lb = 1.0 + 0.1 * torch.randn(64, generator=gen), 0.1 * torch.randn(64, generator=gen)
    if where == "t":
        t[1, 2, 6, 3, 50] = value
    else:
        w[77, 13] = value
    got = of3pair.functional.template_tail(t.to(DEV), lw.to(DEV), lb.to(DEV), w.to(DEV), apply_layer_norm=apply_ln).cpu()
    u = torch.nn.functional.layer_norm(t.double(), (64,), lw.double(), lb.double()) if apply_ln else t.double()
    mean = u.sum(1) / 3
    want = torch.relu(mean) @ w.double().T
    # an output that a large weight makes is off as its input is: sums of three values up to 4, 3 * 2^-24 * 4, of the smallest
    small = float(mean[..., 13][mean[..., 13] > 0].min()) if where == "w" else 1.0
    _same(got, want, rtol=5e-5 + 1e-6 / small)
