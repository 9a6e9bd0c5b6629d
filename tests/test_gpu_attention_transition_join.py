"""The launch that ends the last triangle attention of a block and runs its transition (transition_tiles, AFTER): the bits of the modules by themselves
for one to five position tiles per work-group, hidden slices of 128 and 256, ragged ends, batches; masks on either module or none, in
place; a tensor whose rows are not contiguous and blocks that begin with the attention, where the two stay apart."""
import pytest
import torch

import test_gpu_block_call as blocks
import test_gpu_pass_bf16 as passes

import of3pair

pytestmark = pytest.mark.gpu


# (256 CUs) 1 and 2 tiles: up to 90 and 128 tokens; 4: up to 181, 5: up to 202
@pytest.mark.parametrize("n_mult", [1, 2, 4])
@pytest.mark.parametrize("n,batch", [(1, 1), (30, 3), (90, 1), (91, 1), (128, 1), (64, 4), (179, 1), (202, 1)])
def test_tiles(monkeypatch, n_mult, n, batch):
    passes.test_transition_long_tiles(monkeypatch, n_mult, n, batch)


@pytest.mark.parametrize("n,masked,mask_trans", [(50, False, True), (50, True, False), (100, True, True), (150, True, False)])
def test_masks_and_views(monkeypatch, n, masked, mask_trans):
    m = blocks._fill(of3pair.PairBlock(128, 128, 32, 4), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    z = torch.randn(2, n, n, 128, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(2, n, n, generator=gen) > 0.2).float().to("cuda") if masked else None
    wide = torch.zeros(2, n, n + 3, 128, device="cuda", dtype=torch.bfloat16)
    wide[:, :, :n] = z
    for x in (z, z.transpose(1, 2).contiguous().transpose(1, 2), wide[:, :, :n]):
        want = blocks._by_modules(monkeypatch, lambda: m(x, mask, _mask_trans=mask_trans))
        assert torch.equal(m(x, mask, _mask_trans=mask_trans), want)
        own = x.clone()
        m(own, mask, inplace_safe=True, _mask_trans=mask_trans)
        assert torch.equal(own, want)


@pytest.mark.parametrize("n_mult", [2, 4])
@pytest.mark.parametrize("n,batch", [(1, 2), (45, 1), (60, 4), (91, 1), (127, 2), (181, 1), (182, 1)])
def test_template_tiles(monkeypatch, n_mult, n, batch):
    """64 channels: one tile up to 256 panels, two up to 1024, more work-groups than run at once."""
    m = blocks._fill(of3pair.TemplatePairBlock(64, 16, 64, 4, pair_transition_n=n_mult), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    t = torch.randn(batch, n, n, 64, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float().to("cuda")
    want = blocks._by_modules(monkeypatch, lambda: m(t, mask))
    assert torch.isfinite(want.float()).all()
    assert torch.equal(m(t, mask), want)


@pytest.mark.parametrize("n,batch", [(1, 2), (16, 1), (45, 3), (90, 1), (91, 1), (128, 1), (61, 4), (131, 1), (179, 1), (202, 1), (203, 1)])
def test_with_pair_bias(monkeypatch, n, batch):
    """The pair bias of the attention over s as the end of the same launch: every alignment of a head's runs, ragged ends, one length beyond."""
    m = blocks._fill(of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    s = torch.randn(batch, n, 384, generator=gen).to("cuda").to(torch.bfloat16)
    z = torch.randn(batch, n, n, 128, generator=gen).to("cuda").to(torch.bfloat16)
    tok = (torch.rand(batch, n, generator=gen) > 0.2).float().to("cuda")
    pair = tok[:, :, None] * tok[:, None, :]
    want = blocks._by_modules(monkeypatch, lambda: m(s, z, tok, pair))
    got = m(s, z, tok, pair)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("n_mult", [1, 2, 4, 6])
@pytest.mark.parametrize("n,batch", [(1, 1), (31, 2), (45, 1), (64, 2), (91, 1), (180, 1), (181, 1)])
def test_fp32(monkeypatch, n_mult, n, batch):
    """transition_pass, AFTER, below four tiles of 32 positions per CU, and beyond; hidden slices of 256 (n_mult 1: slices of 128, apart)."""
    m = blocks._fill(of3pair.PairBlock(128, 128, 32, 4, transition_n=n_mult), n).to("cuda").eval()
    gen = torch.Generator().manual_seed(n)
    z = torch.randn(batch, n, n, 128, generator=gen).to("cuda")
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float().to("cuda")
    wide = torch.zeros(batch, n, n + 3, 128, device="cuda")
    wide[:, :, :n] = z
    for x, mk, mask_trans in ((z, mask, True), (z, None, True), (z, mask, False), (wide[:, :, :n], mask, True)):
        want = blocks._by_modules(monkeypatch, lambda: m(x, mk, _mask_trans=mask_trans))
        assert torch.equal(m(x, mk, _mask_trans=mask_trans), want)
    own = z.clone()
    m(own, mask, inplace_safe=True)
    assert torch.equal(own, blocks._by_modules(monkeypatch, lambda: m(z, mask)))


@pytest.mark.parametrize("masked", [True, False])
@pytest.mark.parametrize("n,batch", [(1, 1), (31, 2), (45, 1), (64, 2), (91, 1), (180, 1), (181, 1)])
def test_fp32_with_pair_bias(monkeypatch, n, batch, masked):
    m = blocks._fill(of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4), n).to("cuda").eval()
    gen = torch.Generator().manual_seed(n)
    s, z = torch.randn(batch, n, 384, generator=gen).to("cuda"), torch.randn(batch, n, n, 128, generator=gen).to("cuda")
    tok = (torch.rand(batch, n, generator=gen) > 0.2).float().to("cuda") if masked else torch.ones(batch, n, device="cuda")
    pair = tok[:, :, None] * tok[:, None, :]
    want = blocks._by_modules(monkeypatch, lambda: m(s, z, tok, pair, _mask_trans=masked))
    got = m(s, z, tok, pair, _mask_trans=masked)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
