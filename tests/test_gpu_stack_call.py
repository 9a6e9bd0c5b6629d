"""A stack's call where its pair biases do not fit their room and take turns, and at the lengths of ordinary proteins (whose
first call goes module by module): bit for bit what its blocks give one by one."""
import math

import pytest
import torch

from gpu_util import lib  # noqa: F401

import of3pair
from of3pair import _block

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _stack(dtype, n, no_blocks, heads=16, batch=(1,), c_s=384):
    gen = torch.Generator(device=DEV).manual_seed(51)
    m = of3pair.PairFormerStack(c_s, 128, c_s // heads, heads, 128, 32, 4, no_blocks=no_blocks)
    with torch.no_grad():
        for name, p in m.to(DEV).named_parameters():
            if p.dim() == 2:
                p.copy_(torch.randn(p.shape, generator=gen, device=DEV) * p.shape[1] ** -0.5)
            else:
                p.copy_((1.0 if name.endswith("weight") else 0.0) + 0.1 * torch.randn(p.shape, generator=gen, device=DEV))
    s, z = torch.randn(*batch, n, c_s, generator=gen, device=DEV), torch.randn(*batch, n, n, 128, generator=gen, device=DEV)
    tok = (torch.arange(n, device=DEV) < n - n // 9).float().expand(*batch, n)
    return m.to(dtype).eval(), s.to(dtype), z.to(dtype), tok, tok[..., :, None] * tok[..., None, :]


def _recorded(monkeypatch):
    calls = []
    inner = _block._call
    monkeypatch.setattr(_block, "_call", lambda fn, what, *a: (calls.append(what), inner(fn, what, *a))[1])
    return calls


# one bias at a time (above 64 MB, above 32), two, three, five for seven blocks
@pytest.mark.parametrize("dtype,n,no_blocks,heads,batch,c_s,buffers", [
    (torch.float32, 520, 3, 64, (), 512, 1), (torch.float32, 400, 5, 64, (), 512, 1), (torch.float32, 340, 5, 64, (), 512, 2),
    (torch.float32, 215, 6, 48, (2,), 384, 3), (torch.bfloat16, 512, 7, 24, (1,), 384, 5), (torch.bfloat16, 300, 6, 24, (6,), 384, 2)])
def test_pair_biases_take_turns(monkeypatch, dtype, n, no_blocks, heads, batch, c_s, buffers):
    lib()
    bias = math.prod(batch) * heads * n * n * dtype.itemsize
    assert max(1, (64 << 20) // bias) == buffers < no_blocks
    calls = _recorded(monkeypatch)
    m, s, z, tok, pair = _stack(dtype, n, no_blocks, heads, batch, c_s)
    want = (s, z)
    for blk in m.blocks:
        want = blk(*want, tok, pair)
    m(s, z, tok, pair)
    del calls[:]
    for _ in range(3):
        got = m(s, z, tok, pair)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    a, b = s.clone(), z.clone()
    m(a, b, tok, pair, inplace_safe=True)
    assert torch.equal(a, want[0]) and torch.equal(b, want[1])
    assert calls == ["of3_pairformer_stack_fwd"] * 4


# room for every bias: s of two blocks goes together as long as two more follow, of the last two or three each by itself
@pytest.mark.parametrize("dtype,n", [(torch.bfloat16, 24), (torch.bfloat16, 131), (torch.float32, 40)])
@pytest.mark.parametrize("no_blocks", [1, 2, 3, 4, 5, 6, 9])
def test_single_representation_of_two_blocks_together(monkeypatch, dtype, n, no_blocks):
    lib()
    calls = _recorded(monkeypatch)
    m, s, z, tok, pair = _stack(dtype, n, no_blocks)
    print("stack", dtype, n, no_blocks, flush=True)
    want = (s, z)
    for blk in m.blocks:
        want = blk(*want, tok, pair)
    m(s, z, tok, pair)
    del calls[:]
    for _ in range(3):
        got = m(s, z, tok, pair)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    a, b = s.clone(), z.clone()
    m(a, b, tok, pair, inplace_safe=True)
    assert torch.equal(a, want[0]) and torch.equal(b, want[1])
    assert calls == ["of3_pairformer_stack_fwd"] * 4
