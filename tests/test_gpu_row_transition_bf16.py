"""The bf16 transition of the single representation at row counts around its 32-row tiles, every number of hidden slices of the output kernel.
Tolerance: LayerNorm, hidden activations and result are rounded to bf16 (2^-9 each), as in the tests of the pair transition."""
import pytest
import torch

import test_gpu_transition as tr
from gpu_util import lib
from oracle import pairstack_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n_mult,masked", [(1, 1, False), (31, 2, True), (33, 3, False), (64, 4, True), (97, 4, True), (700, 2, False)])
def test_row_transition(rows, n_mult, masked):
    lib()
    gen = torch.Generator().manual_seed(5600 + rows)
    p = tr._round(orc.make_transition_params(gen, 384, n_mult))
    x = orc.round_bf16(torch.randn(rows, 384, generator=gen) * 1.5 + 0.2)
    mask = (torch.rand(rows, generator=gen) > 0.3).float() if masked else None
    m = tr._module(384, n_mult, p, torch.bfloat16)
    print("row transition bf16", rows, n_mult, masked, flush=True)
    xg, mg = x.to(tr.DEV).to(torch.bfloat16), None if mask is None else mask.to(tr.DEV)
    want = orc.transition_update(x, mask, p)
    floor = orc.transition_update(x.to(torch.bfloat16), None if mask is None else mask.to(torch.bfloat16), tr._bf16(p))
    tr._check("update", m(xg, mask=mg), want, bf16_ref=floor)
    tr._check("x + update", m(xg, mask=mg, _add_residual=True, _inplace=True), x + want, rms_rel=4e-3)
