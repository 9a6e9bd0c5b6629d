"""fp32 products on two fp16 terms: what their scales have to take.  Parameters and LayerNorms far from 1 (a bound follows
from the parameters alone), masks that are no 0 / 1, logits that rise far above those of the first key tile or lie far
below 0, rows that may not be read 16 bytes at a time (another path, another split of the same weights)."""
import pytest
import torch

from gpu_util import lib, report  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"
# as the other fp32 tests of these modules: 1e-5 of the largest value is some 100 roundings of it
REL = 1e-5


def _scaled(p, weights, norms, spread):
    """Every matrix times `weights`, every LayerNorm times `norms`, one channel in 16 of these times `spread`."""
    out = {}
    for name, v in p.items():
        if v.dim() == 2:
            out[name] = v * weights
        else:
            out[name] = v * norms
            out[name][3::16] *= spread
    return out


def _module(cls, p, *args, **kwargs):
    m = cls(*args, **kwargs)
    m.load_state_dict(p, strict=True)
    return m.to(DEV).eval()


def _f64(p):
    return {k: v.double() for k, v in p.items()}


def _no_worse_than_fp32(got, want, plain):
    """The whole result (REL alone is some 70 times the kernels' error): no further off than fp32 arithmetic on the same values."""
    def error(x):
        return float((x.double() - want).norm() / want.norm())

    print("relative 2-norm %.3e, plain fp32 %.3e" % (error(got), error(plain)), flush=True)
    assert error(got) <= error(plain)


SCALES = [(1.0, 1.0, 30.0), (1e-4, 1.0, 1.0), (30.0, 0.1, 1.0), (0.02, 50.0, 1.0), (1e12, 1e-12, 1.0)]


@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("weights,norms,spread", SCALES)
def test_trimul_scales(c, weights, norms, spread):
    lib()
    gen = torch.Generator().manual_seed(8100 + c)
    z = orc.make_pair_input(8101, (1,), 45, c)
    mask = torch.tensor([0.0, 0.25, 1.0, 200.0])[torch.randint(0, 4, (1, 45, 45), generator=gen)]
    p = _scaled(orc.make_trimul_params(gen, c, c), weights, norms, spread)
    print("trimul", c, weights, norms, spread, flush=True)
    want = orc.trimul_update(z.double(), mask.double(), _f64(p), True)
    got = _module(of3pair.TriangleMultiplicationOutgoing, p, c, c)(z.to(DEV), mask.to(DEV)).cpu()
    report("update", got, want, atol=REL * float(want.abs().max()))
    _no_worse_than_fp32(got, want, orc.trimul_update(z, mask, p, True))


@pytest.mark.parametrize("c,d", [(64, 16), (128, 32)])
@pytest.mark.parametrize("weights,norms,spread", [s for s in SCALES if s[0] * s[1] <= 1.0])
def test_triattn_scales(c, d, weights, norms, spread):
    lib()
    gen = torch.Generator().manual_seed(8200 + c)
    z = orc.make_pair_input(8201, (1,), 45, c)
    mask = (torch.rand(1, 45, 45, generator=gen) > 0.2).float()
    p = orc.make_triattn_params(gen, c, d, c // d)
    spread = min(spread, 4.0)  # the logits grow with its square, and the weights' error with the logits
    p = _scaled(p, weights, norms, spread)
    print("triattn", c, d, weights, norms, spread, flush=True)
    want = orc.triattn_update(z.double(), mask.double(), _f64(p), c // d)
    got = _module(of3pair.TriangleAttention, p, c, d, c // d)(z.to(DEV), mask.to(DEV)).cpu()
    report("update", got, want, atol=4 * REL * float(want.abs().max()))
    _no_worse_than_fp32(got, want, orc.triattn_update(z, mask, p, c // d))


@pytest.mark.parametrize("c,n_mult", [(64, 2), (128, 4)])
@pytest.mark.parametrize("weights,norms,spread", SCALES)
def test_transition_scales(c, n_mult, weights, norms, spread):
    lib()
    gen = torch.Generator().manual_seed(8300 + c)
    z = orc.make_pair_input(8301, (1,), 45, c)
    p = _scaled(orc.make_transition_params(gen, c, n_mult), weights, norms, spread)
    print("transition", c, n_mult, weights, norms, spread, flush=True)
    want = orc.transition_update(z.double(), None, _f64(p))
    got = _module(of3pair.SwiGLUTransition, p, c, n_mult)(z.to(DEV)).cpu()
    report("update", got, want, atol=REL * float(want.abs().max()))
    _no_worse_than_fp32(got, want, orc.transition_update(z, None, p))


@pytest.mark.parametrize("c,d", [(64, 16), (128, 32)])
@pytest.mark.parametrize("step", [6.0, 25.0, 60.0, -60.0, 300.0])
@pytest.mark.parametrize("n", [70, 131])
def test_triattn_logits_between_key_tiles(n, c, d, step):
    """The triangle bias of key tile t is about t * step: the weights of the first pass leave the range of fp16 (raised in
    the pass), that of fp32 (second pass), or fall to nothing beside those of the first tile."""
    lib()
    gen = torch.Generator().manual_seed(8400 + c + n)
    z = orc.make_pair_input(8401, (1,), n, c)
    z[..., 0] = 0.0
    z[..., 1] = 0.0
    tile = torch.arange(n) // 32
    z[..., 0] += 20.0 * tile  # channel 0 along k, LayerNorm keeps its order
    p = orc.make_triattn_params(gen, c, d, c // d)
    x = orc.layer_norm(z, p["layer_norm.weight"], p["layer_norm.bias"])[0, :, :, 0].mean(0)
    name = [k for k in p if p[k].dim() == 2 and p[k].shape[0] == c // d][0]
    gap = float(x[32:64].mean() - x[:32].mean())
    p[name] = p[name] * 0.1
    p[name][:, 0] = step / gap
    mask = torch.ones(1, n, n)
    mask[:, 5, : n // 2] = 0.0
    print("triattn tiles", n, c, d, step, flush=True)
    want = orc.triattn_update(z.double(), mask.double(), _f64(p), c // d)
    got = _module(of3pair.TriangleAttention, p, c, d, c // d)(z.to(DEV), mask.to(DEV)).cpu()
    # a logit of size L is held to some 2^-24 L, its weight to as much of itself
    report("update", got, want, atol=(REL + abs(step) * n / 32 * 2.0**-22) * float(want.abs().max()))


@pytest.mark.parametrize("c", [64, 128])
def test_rows_off_16_bytes(c):
    """A block on tensors that start 4 bytes past a 16-byte boundary, against the same values on one."""
    lib()
    n, heads = 37, 4
    gen = torch.Generator().manual_seed(8500 + c)
    p = orc.make_block_params(8501, c, c, c // heads, heads)
    m = _module(of3pair.PairStack, p, c, c, c // heads, heads)
    z = torch.randn(1, n, n, c, generator=gen).to(DEV)
    off = torch.empty(z.numel() + 1, device=DEV)[1:].view(z.shape)
    off.copy_(z)
    print("rows off 16 bytes", c, flush=True)
    mask = (torch.rand(1, n, n, generator=gen) > 0.2).float().to(DEV)
    want = m(z, mask)
    report("block", m(off, mask), want, atol=REL * float(want.abs().max()))
