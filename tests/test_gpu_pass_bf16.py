"""bf16 position-wise passes around the lines of their dispatch: tiles of 32 positions for short sequences, of 128 for the
others, weights as they are (the stages) or in operand order (a block's call)."""
import pytest
import torch

import test_gpu_stages as stages
import test_gpu_block_call as blocks
import test_gpu_transition as transition
from gpu_util import lib  # noqa: F401

import of3pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [(1, 1), (31, 2), (33, 1), (64, 1), (96, 1), (41, 3)])
@pytest.mark.parametrize("c,d", [(128, 32), (64, 16)])
def test_stages(c, d, n, batch):
    for flag in (False, True):
        stages.test_trimul_proj(flag, c, n, batch)
        stages.test_trimul_out(int(flag), c, n, batch)
        stages.test_triattn_proj(flag, c, d, n, batch)
        stages.test_triattn_out(flag, int(flag), c, d, n, batch)


@pytest.mark.parametrize("c,d,n", [(128, 32, 32), (128, 32, 65), (128, 32, 85), (128, 32, 86), (128, 32, 128), (128, 32, 129),
                                   (64, 16, 33), (64, 16, 90), (64, 16, 91)])
def test_packed_weights(monkeypatch, c, d, n):
    """Bit for bit the same however the weights are laid out."""
    lib()
    m = blocks._fill(of3pair.PairStack(c, c, d, 4), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    z = torch.randn(1, n, n, c, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(1, n, n, generator=gen) > 0.2).float().to("cuda")
    want = blocks._by_modules(monkeypatch, lambda: m(z, mask))
    assert torch.equal(m(z, mask), want)


@pytest.mark.parametrize("c,n_mult", [(128, 4), (128, 1), (128, 3), (64, 2), (64, 4)])
@pytest.mark.parametrize("n,batch", [(2, 1), (7, 2), (33, 1), (64, 2), (90, 2), (91, 1), (141, 1)])
def test_transition_tiles(c, n_mult, n, batch):
    transition.test_transition_module(c, n_mult, n, (batch,))


@pytest.mark.parametrize("n_mult", [1, 4])
@pytest.mark.parametrize("n,batch", [(257, 1), (259, 1), (300, 1), (182, 2), (263, 2)])
def test_transition_last_round(n_mult, n, batch):
    """Whole rounds of 256-position tiles and their rest on shorter ones: the second element of a batch, a last tile that
    is not full, and (300, and 256-position tiles in whole rows of another stride) calls that stay in one piece.  The same
    bits as the rows of the tensor one by one."""
    lib()
    gen = torch.Generator().manual_seed(n)
    m = blocks._fill(of3pair.layers.SwiGLUTransition(128, n_mult), n).to("cuda").to(torch.bfloat16).eval()
    x = torch.randn(batch, n, n, 128, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float().to("cuda")
    got = m(x, mask=mask)
    wide = torch.zeros(batch, n, n + 1, 128, device="cuda", dtype=torch.bfloat16)
    wide[:, :, :n] = x
    assert torch.equal(got, m(wide[:, :, :n], mask=mask))
    small = torch.zeros(1, 8, 8, 128, device="cuda", dtype=torch.bfloat16)
    small.view(-1, 128)[:64] = x[-1, -1, -64:]
    small_mask = mask[-1, -1, -64:].reshape(1, 8, 8)
    assert torch.equal(got[-1, -1, -64:], m(small, mask=small_mask).view(-1, 128))


def test_transition_last_round_packed(monkeypatch):
    """The same inside a block's call (weights in operand order, two short tiles per CU)."""
    blocks.test_pairformer_stack(monkeypatch, torch.bfloat16, 260, 1)


@pytest.mark.parametrize("c,d", [(128, 32), (64, 16)])
@pytest.mark.parametrize("n,batch,masked", [(1, 1, False), (2, 3, True), (31, 2, True), (32, 4, False), (33, 2, True), (64, 2, True),
                                            (65, 1, False), (86, 1, True)])
def test_shared_pass(monkeypatch, c, d, n, batch, masked):
    """A block's call at the lengths where the triangle multiplication ends and the attention begins in one pass (and one
    beyond): the bits of the modules, for batches, ragged panels, in place and on a transposed tensor."""
    lib()
    m = blocks._fill(of3pair.PairStack(c, c, d, 4), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    z = torch.randn(batch, n, n, c, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float().to("cuda") if masked else None
    want = blocks._by_modules(monkeypatch, lambda: m(z, mask))
    assert torch.isfinite(want.float()).all()
    assert torch.equal(m(z, mask), want)
    own = z.clone()
    m(own, mask, inplace_safe=True)
    assert torch.equal(own, want)
    zt = z.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(m(zt, mask), want)


@pytest.mark.parametrize("n_mult", [1, 4])
@pytest.mark.parametrize("n,batch", [(129, 1), (150, 1), (104, 2), (181, 1), (182, 1), (202, 1), (203, 1)])
def test_transition_long_tiles(monkeypatch, n_mult, n, batch):
    """Inside a block's call: tiles of 128 positions up to four panels of 32 per CU, of 160 up to five, and one beyond
    (256 CUs; 104: two elements, each with a tile that is not full)."""
    lib()
    m = blocks._fill(of3pair.PairBlock(128, 128, 32, 4, transition_n=n_mult), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    z = torch.randn(batch, n, n, 128, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float().to("cuda")
    want = blocks._by_modules(monkeypatch, lambda: m(z, mask))
    assert torch.isfinite(want.float()).all()
    assert torch.equal(m(z, mask), want)
