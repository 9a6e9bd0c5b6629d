"""A method or function that a caller has put in the place of one a block run module by module calls, is called: the block
does not go through one library call then."""
import pytest
import torch

from gpu_util import lib  # noqa: F401

import of3pair
from of3pair import _block
from of3pair import functional as F3

pytestmark = pytest.mark.gpu
DEV = "cuda"
CLASSES = [(of3pair.PairBlock, "forward"), (of3pair.AttentionPairBias, "forward"), (of3pair.SwiGLUTransition, "forward"),
           (of3pair.PairFormerBlock, "forward"), (of3pair.PairBlock, "tri_mul_out_in"), (of3pair.PairStack, "tri_att_start_end"),
           (of3pair.TriangleMultiplicationIncoming, "_weights"), (torch.nn.Module, "__call__"),
           (F3, "triangle_attention"), (F3, "swiglu_transition"), (F3, "pair_bias")]
INSTANCES = [("pair_stack", "tri_mul_out_in"), ("pair_stack", "tri_att_start_end"), ("pair_stack", "forward"),
             ("pair_stack.tri_mul_out", "_weights"), ("pair_stack.pair_transition", "forward"), ("single_transition", "forward"),
             ("attn_pair_bias", "_compiled_call_impl")]


def _setup(monkeypatch, n=21):
    lib()
    torch.manual_seed(41)
    m = of3pair.PairFormerStack(384, 128, 24, 16, 128, 32, 4, no_blocks=2)
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 2:
                p.normal_(std=p.shape[1] ** -0.5)
    m = m.to(DEV).to(torch.bfloat16).eval()
    s, z = torch.randn(1, n, 384, device=DEV).to(torch.bfloat16), torch.randn(1, n, n, 128, device=DEV).to(torch.bfloat16)
    want = m(s, z, None, None)
    calls = []
    inner = _block._call
    monkeypatch.setattr(_block, "_call", lambda fn, what, *a: (calls.append(what), inner(fn, what, *a))[1])

    def run():
        del calls[:]
        got = m(s, z, None, None)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        return list(calls)

    assert run() == ["of3_pairformer_stack_fwd"]
    return m, run


def _recording(monkeypatch, owner, name, seen, instance=False):
    inner = getattr(owner, name)
    if inner is None:  # a module that torch.compile has not been asked for
        inner = owner._call_impl

    def put(*args, **kwargs):
        seen.append(name)
        return inner(*args, **kwargs)

    monkeypatch.setattr(owner, name, put, raising=not instance)


@pytest.mark.parametrize("owner,name", CLASSES, ids=lambda v: getattr(v, "__name__", v))
def test_replaced_on_the_class(monkeypatch, owner, name):
    m, run = _setup(monkeypatch)
    seen = []
    with monkeypatch.context() as mp:
        _recording(mp, owner, name, seen)
        assert run() == [] and seen
    assert run() == ["of3_pairformer_stack_fwd"]


@pytest.mark.parametrize("path,name", INSTANCES)
def test_replaced_on_an_instance(monkeypatch, path, name):
    m, run = _setup(monkeypatch)
    seen = []
    own = m.blocks[1].get_submodule(path)
    _recording(monkeypatch, own, name, seen, instance=True)
    assert "of3_pairformer_stack_fwd" not in run() and len(seen) == 1
    del own.__dict__[name]
    assert run() == ["of3_pairformer_stack_fwd"]


@pytest.mark.parametrize("path,name", [("pair_stack", "tri_att_start_end"), ("single_transition", "forward"), ("attn_pair_bias", "forward"),
                                       ("pair_stack.tri_mul_in", "_weights")])
def test_another_class_given_to_an_instance(monkeypatch, path, name):
    m, run = _setup(monkeypatch)
    own, seen = m.blocks[0].get_submodule(path), []
    kind = type(own)

    def put(self, *args, **kwargs):
        seen.append(name)
        return getattr(kind, name)(self, *args, **kwargs)

    own.__class__ = type("Other", (kind,), {name: put})
    assert "of3_pairformer_stack_fwd" not in run() and len(seen) == 1
    own.__class__ = kind
    assert run() == ["of3_pairformer_stack_fwd"]


class _Wrapped(torch.nn.Linear):
    pass


def _own_class(m):
    lin = m.blocks[0].pair_stack.tri_att_end.mha.linear_v
    lin.__class__ = _Wrapped
    return lambda: setattr(lin, "__class__", torch.nn.Linear)


def _wrapped(m):
    t = m.blocks[1].single_transition
    lin = t.linear_out
    t.linear_out = _Wrapped(lin.in_features, lin.out_features, bias=False).to(lin.weight)
    t.linear_out.weight = lin.weight
    return lambda: setattr(t, "linear_out", lin)


def _parametrized(m):
    mul = m.blocks[0].pair_stack.tri_mul_in
    torch.nn.utils.parametrize.register_parametrization(mul.linear_b_g, "weight", torch.nn.Identity())
    return lambda: torch.nn.utils.parametrize.remove_parametrizations(mul.linear_b_g, "weight")


def _other_inf(m):
    m.blocks[1].pair_stack.tri_att_start.inf = 2e9
    return lambda: setattr(m.blocks[1].pair_stack.tri_att_start, "inf", 1e9)


def _no_head_width(m):
    q = m.blocks[0].attn_pair_bias.mha
    lin = q.linear_q
    del q.linear_q
    q.linear_q = torch.nn.Identity()
    q.linear_q.weight, q.linear_q.bias = lin.weight, lin.bias
    return lambda: setattr(q, "linear_q", lin)


@pytest.mark.parametrize("change", [_own_class, _wrapped, _parametrized, _other_inf, _no_head_width])
def test_a_refused_block_is_served_once_it_is_restored(monkeypatch, change):
    m, run = _setup(monkeypatch)
    _block._plans.clear()
    restore = change(m)
    for _ in range(3):
        assert "of3_pairformer_stack_fwd" not in run()
    restore()
    run()
    assert run() == ["of3_pairformer_stack_fwd"]


@pytest.mark.parametrize("n", [30, 310])
def test_widths_of_s_are_refused_as_by_the_modules(n):
    """A batch of single representations has 384 channels; one without a batch has any.  The first call of a block, the
    second and a stack's own agree."""
    lib()
    m = of3pair.PairFormerStack(64, 64, 16, 4, 64, 16, 4, no_blocks=2).to(DEV).eval()
    s, z = torch.randn(n, 64, device=DEV), torch.randn(n, n, 64, device=DEV)
    for _ in range(3):
        with pytest.raises(ValueError):
            m(s[None], z[None], None, None)
    want = m(s, z, None, None)
    for _ in range(2):
        got = m(s, z, None, None)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        with pytest.raises(ValueError):
            m(s[None], z[None], None, None)


def test_a_refused_block_with_another_weight(monkeypatch):
    """A block refused over a parameter's shape is compared by that parameter, not by its values."""
    m, run = _setup(monkeypatch)
    a = m.blocks[0].attn_pair_bias
    weight, bias, heads = a.mha.linear_q.weight, a.mha.linear_q.bias, a.no_heads
    a.no_heads = 5  # 384 channels are no five heads
    with pytest.raises(ValueError):
        run()
    a.mha.linear_q.weight = torch.nn.Parameter(weight.detach().clone())
    with pytest.raises(ValueError):
        run()
    a.no_heads = heads
    run()
    assert run() == ["of3_pairformer_stack_fwd"]
    a.mha.linear_q.weight, a.mha.linear_q.bias = weight, bias
    assert run() == ["of3_pairformer_stack_fwd"]
