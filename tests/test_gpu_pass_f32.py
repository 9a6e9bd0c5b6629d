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
