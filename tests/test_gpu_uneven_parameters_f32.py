"""fp32 modules on two fp16 terms with parameters of uneven size, as training leaves them: a LayerNorm weight s times the others
with the columns behind it s times smaller, a hidden or value channel s times larger whose next column makes up for it, gates
that are nearly closed.  The values that a scale from a loose bound would push to fp16's last bits are then as large a
part of the result as any.

The bound is plain fp32's own error on the same values: what the products here add up, in fp32 too, leaves 0.3 to 0.8 of it."""
import pytest
import torch

from gpu_util import lib  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _closed_gates(p, norm, gates, by):
    """Every gate's argument lower by `by`."""
    b = p[_name(p, norm).replace(".weight", ".bias")]
    if by:
        b += 1.0
    for name in gates:
        p[_name(p, name)] -= by * b / b.pow(2).sum()


def _name(p, *parts):
    names = [k for k in p if k.endswith(".weight") and all(q in k for q in parts)]
    assert len(names) == 1, (parts, names)
    return names[0]


def _norm_channel(p, norm, behind, s, channel=3):
    p[_name(p, norm)][channel] *= s
    for name in behind:
        p[_name(p, name)][:, channel] /= s


def _check(what, module, args, oracle, p, beyond=0.0):
    want = oracle(*[a.double() for a in args], {k: v.double() for k, v in p.items()})
    plain = oracle(*args, p)
    module.load_state_dict(p, strict=True)
    got = module.to(DEV).eval()(*[a.to(DEV) for a in args]).cpu()

    def error(x):
        return float((x.double() - want).norm() / max(float(want.norm()), 1e-30))

    print("%s: relative 2-norm %.3e, plain fp32 %.3e" % (what, error(got), error(plain)), flush=True)
    assert got.isfinite().all()
    assert error(got) <= error(plain) + beyond


@pytest.mark.parametrize("c,n_mult", [(64, 2), (64, 4), (128, 4)])
@pytest.mark.parametrize("s,rows", [(1, 1), (30, 1), (100, 1), (300, 1), (1, 30), (1, 100), (1, 1000), (30, 10)])
def test_transition_uneven(c, n_mult, s, rows):
    lib()
    gen = torch.Generator().manual_seed(8800 + c)
    p = orc.make_transition_params(gen, c, n_mult)
    _norm_channel(p, "layer_norm", ("linear_a", "linear_b"), s)
    for hidden in (5, 6, 70):
        p[_name(p, "linear_a")][hidden] *= rows
        p[_name(p, "linear_b")][hidden] *= rows
        p[_name(p, "linear_out")][:, hidden] /= rows**2
    z = orc.make_pair_input(8801, (1,), 45, c)
    _check("transition %d x %d, norm %d, rows %d" % (c, n_mult, s, rows), of3pair.SwiGLUTransition(c, n_mult), [z],
           lambda x, q: orc.transition_update(x, None, q), p)


@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("s,rows,closed", [(1, 1, 0.0), (30, 1, 0.0), (300, 1, 0.0), (1, 100, 0.0), (1, 1, 9.0), (30, 1, 9.0)])
def test_trimul_uneven(c, s, rows, closed):
    lib()
    gen = torch.Generator().manual_seed(8810 + c)
    p = orc.make_trimul_params(gen, c, c)
    _closed_gates(p, "layer_norm_in", ("linear_a_g", "linear_b_g"), closed)
    _norm_channel(p, "layer_norm_in", ("linear_a_p", "linear_a_g", "linear_b_p", "linear_b_g", "linear_g"), s)
    p["linear_a_p.weight"][7] *= rows
    p["linear_b_p.weight"][7] /= rows
    z = orc.make_pair_input(8811, (1,), 45, c)
    mask = torch.ones(1, 45, 45)
    _check("trimul %d, norm %d, rows %d, closed %g" % (c, s, rows, closed), of3pair.TriangleMultiplicationOutgoing(c, c), [z, mask],
           lambda x, m, q: orc.trimul_update(x, m, q, True), p)


@pytest.mark.parametrize("c,d", [(64, 16), (128, 32)])
@pytest.mark.parametrize("s,rows,closed", [(1, 1, 0.0), (30, 1, 0.0), (300, 1, 0.0), (1, 100, 0.0), (1, 3000, 0.0), (30, 1, 9.0)])
def test_triattn_uneven(c, d, s, rows, closed):
    lib()
    gen = torch.Generator().manual_seed(8820 + c)
    heads = c // d
    p = orc.make_triattn_params(gen, c, d, heads)
    _closed_gates(p, "layer_norm", ("linear_g",), closed)
    _norm_channel(p, "layer_norm", ("linear_q", "linear_k", "linear_v", "linear_g", "linear_z"), s)
    p[_name(p, "linear_v")][9] *= rows
    p[_name(p, "linear_o")][:, 9] /= rows
    z = orc.make_pair_input(8821, (1,), 45, c)
    mask = torch.ones(1, 45, 45)
    _check("triattn %d, norm %d, rows %d, closed %g" % (c, s, rows, closed), of3pair.TriangleAttention(c, d, heads), [z, mask],
           lambda x, m, q: orc.triattn_update(x, m, q, heads), p)


ZERO = {
    "transition": ("layer_norm.weight", "layer_norm.bias", "linear_a.weight", "linear_b.weight", "linear_out.weight"),
    "trimul": ("layer_norm_in.weight", "linear_a_p.weight", "linear_b_g.weight", "linear_z.weight"),
    "triattn": ("layer_norm.weight", "layer_norm.bias", "linear_q.weight", "linear_v.weight", "linear_o.weight"),
}


@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("part", ["whole", "rows"])
@pytest.mark.parametrize("kind,name", [(k, n) for k in ZERO for n in ZERO[k]])
def test_zero_parameters(kind, name, part, c):
    """A whole parameter of zeros, or its first 32 rows (a tile of them) and some others."""
    lib()
    gen = torch.Generator().manual_seed(8830 + c)
    z = orc.make_pair_input(8831, (1,), 37, c)
    mask = torch.ones(1, 37, 37)
    if kind == "transition":
        p, m, args = orc.make_transition_params(gen, c, 2), of3pair.SwiGLUTransition(c, 2), [z]
        oracle = lambda x, q: orc.transition_update(x, None, q)  # noqa: E731
    elif kind == "trimul":
        p, m, args = orc.make_trimul_params(gen, c, c), of3pair.TriangleMultiplicationOutgoing(c, c), [z, mask]
        oracle = lambda x, k, q: orc.trimul_update(x, k, q, True)  # noqa: E731
    else:
        p, m, args = orc.make_triattn_params(gen, c, c // 4, 4), of3pair.TriangleAttention(c, c // 4, 4), [z, mask]
        oracle = lambda x, k, q: orc.triattn_update(x, k, q, 4)  # noqa: E731
    v = p[[k for k in p if k.endswith(name)][0]]
    if part == "whole":
        v.zero_()
    else:
        v[:32] = 0
        v[33::7] = 0
    _check("%s, zeros in %s (%s)" % (kind, name, part), m, args, oracle, p)


@pytest.mark.parametrize("n", [45, 150])  # the attention's end with the transition's launch, and by itself
@pytest.mark.parametrize("rows", [1, 1000])
def test_block_uneven(n, rows):
    """A whole block: value channels and hidden channels of every tile of 32 columns at another size."""
    lib()
    gen = torch.Generator().manual_seed(8840)
    p = orc.make_block_params(8841, 128, 128, 32, 4)
    p.update({"pair_transition." + k: v for k, v in orc.make_transition_params(gen, 128, 4).items()})
    for k in list(p):
        for one, following in (("mha.linear_v", "mha.linear_o"), ("swiglu.linear_b", "linear_out")):
            if one in k:
                size = rows ** torch.linspace(-1, 1, p[k].shape[0] // 32).repeat_interleave(32)
                p[k] = p[k] * size[:, None]
                p[k.replace(one, following)] = p[k.replace(one, following)] / size
    z = orc.make_pair_input(8842, (1,), n, 128)
    mask = torch.ones(1, n, n)
    _check("block %d, rows %d" % (n, rows), of3pair.PairBlock(128, 128, 32, 4, "swiglu", 4, 0.25, False, 1e9), [z, mask],
           lambda x, m, q: orc.pair_block(x, m, q, 4), p)
