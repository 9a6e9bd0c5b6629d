"""The fp32 kernels of the single representation on the matrix instructions, at the edges of their tiles: row
counts around the 32-row tile, the smallest and largest channel counts that they serve (a wave without a block of
inputs, four blocks per wave), every head width, keys past the last tile, rows whose keys are all masked."""
import pytest
import torch

from gpu_util import lib, report  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,c_s,c_head,heads,mask", [
    (1, 32, 8, 4, None), (31, 64, 32, 1, "tail"), (32, 96, 24, 4, "all"), (33, 160, 16, 10, "tail"), (65, 384, 24, 16, "tail"),
    (130, 512, 32, 16, None), (132, 512, 8, 64, "tail")])
def test_attention_pair_bias_fp32_tiles(n, c_s, c_head, heads, mask):
    lib()
    gen = torch.Generator().manual_seed(5200 + n)
    p = orc.make_attention_pair_bias_params(gen, c_s, 32, c_head, heads)
    a = torch.randn(1, n, c_s, generator=gen) * 1.5 + 0.2
    z = orc.make_pair_input(5300 + n, (1,), n, 32)
    m = None
    if mask:
        m = torch.ones(1, n)
        m[..., 0 if mask == "all" else n - max(1, n // 3):] = 0
    mod = of3pair.AttentionPairBias(c_s, c_s, c_s, c_s, 32, c_head, heads)
    mod.load_state_dict(p, strict=True)
    mod = mod.to(DEV).eval()
    print("attention pair bias fp32", n, c_s, c_head, heads, mask, flush=True)
    ag, zg, mg = a.to(DEV), z.to(DEV), None if m is None else m.to(DEV)
    want = orc.attention_pair_bias(a, z, m, p, heads)
    scale = max(1.0, float(want.abs().max()))
    report("update", mod(ag, zg, mask=mg).cpu(), want, atol=5e-6 * scale)
    got = mod(ag, zg, mask=mg, _add_residual=True, _inplace=True)
    assert got.data_ptr() == ag.data_ptr()
    report("a + update in place", got.cpu(), a + want, atol=5e-6 * max(scale, float(a.abs().max())))


@pytest.mark.parametrize("rows,c,n_mult,masked", [(1, 32, 1, False), (31, 384, 4, True), (33, 160, 2, True),
                                                  (64, 512, 4, False), (97, 416, 3, True)])
def test_row_transition_fp32_tiles(rows, c, n_mult, masked):
    lib()
    gen = torch.Generator().manual_seed(5400 + rows)
    p = orc.make_transition_params(gen, c, n_mult)
    x = torch.randn(rows, c, generator=gen) * 1.5 + 0.2
    mask = (torch.rand(rows, generator=gen) > 0.3).float() if masked else None
    mod = of3pair.SwiGLUTransition(c, n_mult)
    mod.load_state_dict(p, strict=True)
    mod = mod.to(DEV).eval()
    print("row transition fp32", rows, c, n_mult, masked, flush=True)
    xg, mg = x.to(DEV), None if mask is None else mask.to(DEV)
    want = orc.transition_update(x, mask, p)
    scale = max(1.0, float(want.abs().max()))
    report("update", mod(xg, mask=mg).cpu(), want, atol=5e-6 * scale)
    got = mod(xg, mask=mg, _add_residual=True, _inplace=True)
    assert got.data_ptr() == xg.data_ptr()
    report("x + update in place", got.cpu(), x + want, atol=5e-6 * max(scale, float(x.abs().max())))
