"""The fp32 position-wise passes at 64 and 128 channels: lengths around the 32-position tile and the four-row groups,
more tiles than a round of the persistent grids, both head widths, transposed and batched views, masks."""
import pytest
import torch

from gpu_util import lib, report  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENGTHS = [(1, 2), (31, 1), (33, 3), (66, 1), (131, 1)]


def _inputs(seed, n, batch, c, masked):
    gen = torch.Generator().manual_seed(seed)
    z = orc.make_pair_input(seed + 1, (batch,), n, c)
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float() if masked else None
    return gen, z, mask


@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("n,batch", LENGTHS)
def test_trimul(n, batch, c):
    lib()
    for outgoing in (True, False):
        gen, z, mask = _inputs(6100 + n + c, n, batch, c, masked=outgoing)
        p = orc.make_trimul_params(gen, c, c)
        cls = of3pair.TriangleMultiplicationOutgoing if outgoing else of3pair.TriangleMultiplicationIncoming
        m = cls(c, c)
        m.load_state_dict(p, strict=True)
        m = m.to(DEV).eval()
        print("trimul fp32", n, batch, c, outgoing, flush=True)
        zg, mg = z.to(DEV), None if mask is None else mask.to(DEV)
        want = orc.trimul_update(z, mask, p, outgoing)
        tol = 1e-5 * max(1.0, float(want.abs().max()))
        report("update", m(zg, mg).cpu(), want, atol=tol)
        got = m(zg, mg, inplace_safe=True, _add_with_inplace=True)
        report("z + update in place", got.cpu(), z + want, atol=tol)


@pytest.mark.parametrize("c,d", [(64, 16), (64, 32), (128, 16), (128, 32)])
@pytest.mark.parametrize("n,batch", LENGTHS)
def test_triattn(n, batch, c, d):
    lib()
    for starting in (True, False):
        gen, z, mask = _inputs(6500 + n + c + d, n, batch, c, masked=starting)
        p = orc.make_triattn_params(gen, c, d, c // d)
        m = of3pair.TriangleAttention(c, d, c // d, starting=starting)
        m.load_state_dict(p, strict=True)
        m = m.to(DEV).eval()
        print("triattn fp32", n, batch, c, d, starting, flush=True)
        zg, mg = z.to(DEV), None if mask is None else mask.to(DEV)
        want = orc.triattn_update(z, mask, p, c // d, starting=starting)
        tol = 1e-5 * max(1.0, float(want.abs().max()))
        report("update", m(zg, mg).cpu(), want, atol=tol)
        report("x + update", m(zg, mg, _add_residual=True).cpu(), z + want, atol=tol)


@pytest.mark.parametrize("c,n_mult", [(64, 2), (64, 4), (128, 1), (128, 2), (128, 4), (128, 6)])
@pytest.mark.parametrize("n,batch", LENGTHS + [(190, 1)])
def test_transition(n, batch, c, n_mult):
    """Hidden slices of 128 and 256, tiles of 32 and 64 positions, flattened and row-by-row views."""
    lib()
    gen, z, mask = _inputs(6900 + n + c + n_mult, n, batch, c, masked=n != 33)
    p = orc.make_transition_params(gen, c, n_mult)
    m = of3pair.SwiGLUTransition(c, n_mult)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).eval()
    print("transition fp32", n, batch, c, n_mult, flush=True)
    zg, mg = z.to(DEV), None if mask is None else mask.to(DEV)
    want = orc.transition_update(z, mask, p)
    tol = 1e-5 * max(1.0, float(want.abs().max()))
    report("update", m(zg, mask=mg).cpu(), want, atol=tol)
    wide = torch.zeros(batch, n, n + 3, c, device=DEV)
    wide[:, :, :n] = zg
    got = m(wide[:, :, :n], mask=mg, _add_residual=True)
    report("x + update of a windowed view", got.cpu(), z + want, atol=tol)
    got = m(zg, mask=mg, _add_residual=True, _inplace=True)
    report("x + update in place", got.cpu(), z + want, atol=tol)


@pytest.mark.parametrize("c,heads,offset", [(64, 1, True), (64, 16, False), (128, 9, True), (128, 16, True), (128, 32, False)])
@pytest.mark.parametrize("n,batch", LENGTHS)
def test_pair_bias(n, batch, c, heads, offset):
    lib()
    gen, z, _ = _inputs(7300 + n + c + heads, n, batch, c, masked=False)
    p = orc.make_pair_bias_params(gen, c, heads, offset)
    m = of3pair.PairBiasProjection(c, heads, create_offset=offset)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).eval()
    print("pair bias fp32", n, batch, c, heads, flush=True)
    want = orc.pair_bias(z, p)
    report("pair bias", m(z.to(DEV)).cpu(), want, atol=1e-5 * max(1.0, float(want.abs().max())))
    zt = z.to(DEV).transpose(1, 2)
    report("pair bias of a transposed view", m(zt).cpu(), orc.pair_bias(z.transpose(1, 2), p),
           atol=1e-5 * max(1.0, float(want.abs().max())))


@pytest.mark.parametrize("n,batch,templates,apply_ln", [(1, 1, 1, True), (7, 2, 3, True), (33, 1, 4, False), (130, 1, 2, True)])
def test_template_tail(n, batch, templates, apply_ln):
    lib()
    from of3pair import functional as F3

    gen = torch.Generator().manual_seed(7700 + n)
    t = torch.randn(batch, templates, n, n, 64, generator=gen)
    w = torch.randn(128, 64, generator=gen) / 8
    lw, lb = 1 + 0.1 * torch.randn(64, generator=gen), 0.1 * torch.randn(64, generator=gen)
    print("template tail fp32", n, batch, templates, apply_ln, flush=True)
    want = orc.template_tail(orc.layer_norm(t, lw, lb) if apply_ln else t, w)
    got = F3.template_tail(t.to(DEV), lw.to(DEV), lb.to(DEV), w.to(DEV), apply_layer_norm=apply_ln)
    report("template tail", got.cpu(), want, atol=1e-5 * max(1.0, float(want.abs().max())))
