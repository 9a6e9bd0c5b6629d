"""Whole blocks through one library call: bit for bit what the same block gives module by module, and changes that a
caller makes to a block between calls are seen (other weights, a replaced submodule, another dtype, a hook)."""
import pytest
import torch

from gpu_util import lib  # noqa: F401

import of3pair
from of3pair import _block

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _fill(m, seed):
    gen = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for name, p in m.named_parameters():
            if p.dim() == 2:
                p.copy_(torch.randn(p.shape, generator=gen) * p.shape[1] ** -0.5)
            else:
                p.copy_((1.0 if name.endswith("weight") else 0.0) + 0.1 * torch.randn(p.shape, generator=gen))
    return m


def _count(monkeypatch):
    """Counts the blocks that go through one call."""
    calls = []
    inner = _block._call
    monkeypatch.setattr(_block, "_call", lambda fn, what, *a: (calls.append(what), inner(fn, what, *a))[1])
    return calls


def _by_modules(monkeypatch, fn):
    with monkeypatch.context() as mp:
        mp.setattr(_block, "_gather", lambda *a: None)
        return fn()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mask_trans,inplace", [(True, False), (False, True)])
def test_pairformer_block(monkeypatch, dtype, mask_trans, inplace):
    lib()
    calls = _count(monkeypatch)
    n = 37
    m = _fill(of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4), 3).to(DEV).to(dtype).eval()
    gen = torch.Generator().manual_seed(4)
    s, z = torch.randn(2, n, 384, generator=gen).to(DEV).to(dtype), torch.randn(2, n, n, 128, generator=gen).to(DEV).to(dtype)
    tok = (torch.rand(2, n, generator=gen) > 0.2).float().to(DEV)
    pair = tok[:, :, None] * tok[:, None, :]

    def run():
        a, b = s.clone(), z.clone()
        out = m(a, b, tok, pair, inplace_safe=inplace, _mask_trans=mask_trans)
        if inplace:
            assert out[0].data_ptr() == a.data_ptr() and out[1].data_ptr() == b.data_ptr()
        else:
            assert torch.equal(a, s) and torch.equal(b, z)
        return out

    want = _by_modules(monkeypatch, run)
    assert not calls
    got = run()
    assert calls == ["of3_pairformer_block_fwd"]
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    # what a caller changes is seen by the next call
    with torch.no_grad():
        m.pair_stack.tri_att_end.mha.linear_v.weight.mul_(2.0)
    m.single_transition.linear_out = _fill(torch.nn.Linear(4 * 384, 384, bias=False), 9).to(DEV).to(dtype)
    m.pair_stack.tri_mul_in.linear_g.weight = torch.nn.Parameter(m.pair_stack.tri_mul_in.linear_g.weight.detach() * 0.5)
    m.attn_pair_bias.inf = 1e4
    want = _by_modules(monkeypatch, run)
    got = run()
    assert len(calls) == 2 and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert not torch.equal(got[0], s)
    # a hook on a submodule, or parameters of another dtype than the activations: module by module
    seen = []
    handle = m.single_transition.register_forward_hook(lambda *a: seen.append(1))
    again = run()
    assert calls[2:] == ["of3_pair_block_fwd"] and seen and torch.equal(again[0], got[0])  # the pair stack has no hook
    handle.remove()
    m.to(torch.float32 if dtype == torch.bfloat16 else torch.bfloat16)
    run()
    assert len(calls) == 3


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_template_pair_block(monkeypatch, dtype, first, fused):
    lib()
    calls = _count(monkeypatch)
    m = of3pair.TemplatePairBlock(64, 16, 64, 4, tri_mul_first=first, fuse_projection_weights=fused)
    m = _fill(m, 5).to(DEV).to(dtype).eval()
    gen = torch.Generator().manual_seed(6)
    z = torch.randn(2, 3, 19, 19, 64, generator=gen).to(DEV).to(dtype)
    mask = (torch.rand(2, 1, 19, 19, generator=gen) > 0.2).float().to(DEV).expand(2, 3, 19, 19)
    want = _by_modules(monkeypatch, lambda: m(z, mask))
    got = m(z, mask)
    assert calls == ["of3_pair_block_fwd"] and torch.equal(got, want)
    zt = z.transpose(-2, -3)  # a transposed view is walked as it is
    want = _by_modules(monkeypatch, lambda: m(zt, mask))
    assert torch.equal(m(zt, mask), want) and len(calls) == 2


def test_pair_stack_without_mask(monkeypatch):
    lib()
    calls = _count(monkeypatch)
    m = _fill(of3pair.PairStack(128, 128, 32, 4), 7).to(DEV).to(torch.bfloat16).eval()
    z = torch.randn(1, 21, 21, 128, generator=torch.Generator().manual_seed(8)).to(DEV).to(torch.bfloat16)
    want = _by_modules(monkeypatch, lambda: m(z, None))
    assert torch.equal(m(z, None), want) and calls == ["of3_pair_block_fwd"]


@pytest.mark.parametrize("dtype,n,no_blocks", [(torch.bfloat16, 40, 1), (torch.bfloat16, 37, 2), (torch.bfloat16, 200, 3), (torch.bfloat16, 24, 9),
                                               (torch.float32, 33, 5)])
def test_pairformer_stack(monkeypatch, dtype, n, no_blocks):
    """A stack's call, its single representation on a second stream, against its blocks one by one; again under a capture."""
    lib()
    calls = _count(monkeypatch)
    m = _fill(of3pair.PairFormerStack(384, 128, 24, 16, 128, 32, 4, no_blocks=no_blocks), 11).to(DEV).to(dtype).eval()
    gen = torch.Generator().manual_seed(12)
    s, z = torch.randn(1, n, 384, generator=gen).to(DEV).to(dtype), torch.randn(1, n, n, 128, generator=gen).to(DEV).to(dtype)
    tok = (torch.rand(1, n, generator=gen) > 0.2).float().to(DEV)
    pair = tok[:, :, None] * tok[:, None, :]
    want = (s, z)
    for blk in m.blocks:
        want = blk(*want, tok, pair)
    del calls[:]
    for _ in range(3):
        got = m(s, z, tok, pair)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    a, b = s.clone(), z.clone()
    m(a, b, tok, pair, inplace_safe=True)
    assert torch.equal(a, want[0]) and torch.equal(b, want[1])
    assert calls == ["of3_pairformer_stack_fwd"] * 4
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        got = m(s, z, tok, pair)
    torch.cuda.current_stream().wait_stream(other)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m(s, z, tok, pair)
    for _ in range(3):
        out[0].zero_(), out[1].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], want[0]) and torch.equal(out[1], want[1])
        m(s, z, tok, pair)
    # blocks of other widths than the first, or a hook on one: block by block
    if no_blocks > 1:
        handle = m.blocks[1].register_forward_hook(lambda *args: None)
        got = m(s, z, tok, pair)
        assert torch.equal(got[0], want[0]) and calls[-1] == "of3_pairformer_block_fwd"
        handle.remove()


def test_stack_captured_after_one_eager_call():
    """The first call of a stack goes block by block, the second, under a capture, through the stack's own call."""
    lib()
    m = _fill(of3pair.PairFormerStack(384, 128, 24, 16, 128, 32, 4, no_blocks=2), 21).to(DEV).to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(22)
    s, z = (torch.randn(*shape, generator=gen).to(DEV).to(torch.bfloat16) for shape in ((1, 45, 384), (1, 45, 45, 128)))
    want = [t.clone() for t in m(s, z, None, None)]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = m(s, z, None, None)
    for _ in range(3):
        out[0].zero_(), out[1].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], want[0]) and torch.equal(out[1], want[1])
        assert all(torch.equal(a, b) for a, b in zip(m(s, z, None, None), want))
