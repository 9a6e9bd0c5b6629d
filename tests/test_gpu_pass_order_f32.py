"""fp32 passes: the two halves of a work-group that take a tile's vector and matrix work in opposite order, at one tile per
work-group, some with two, and several; and rows too far apart for a buffer offset, which the general kernels serve."""
import pytest
import torch

from gpu_util import lib, report  # noqa: F401
from oracle import pairstack_oracle as orc

import of3pair

pytestmark = pytest.mark.gpu
DEV = "cuda"
REL = 1e-5  # of the largest value: some 100 roundings of it, as the other fp32 tests of these modules


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("n", [84, 85, 131, 181])  # 252, 264, 660 and 1104 tiles of 32 positions on 256 CUs
def test_trimul_tiles_per_work_group(n, masked):
    lib()
    c = 128
    gen = torch.Generator().manual_seed(8600 + n)
    z = orc.make_pair_input(8601, (1,), n, c)
    mask = (torch.rand(1, n, n, generator=gen) > 0.2).float() if masked else None
    p = orc.make_trimul_params(gen, c, c)
    m = of3pair.TriangleMultiplicationOutgoing(c, c)
    m.load_state_dict(p, strict=True)
    print("trimul", n, masked, flush=True)
    ones = torch.ones(1, n, n) if mask is None else mask
    want = orc.trimul_update(z.double(), ones.double(), {k: v.double() for k, v in p.items()}, True)
    got = m.to(DEV).eval()(z.to(DEV), None if mask is None else mask.to(DEV)).cpu()
    report("update", got, want, atol=REL * float(want.abs().max()))


@pytest.mark.parametrize("c", [64, 128])
def test_rows_far_apart(c):
    lib()
    n, heads, far = 5, 4, 1 << 24
    p = orc.make_block_params(8602, c, c, c // heads, heads)
    m = of3pair.PairStack(c, c, c // heads, heads)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).eval()
    z = torch.randn(1, n, n, c, generator=torch.Generator().manual_seed(8603)).to(DEV)
    apart = torch.zeros(n * far, device=DEV).as_strided((1, n, n, c), (n * far, far, c, 1))
    apart.copy_(z)
    mask = torch.ones(1, n, n, device=DEV)
    print("rows far apart", c, flush=True)
    want = m(z, mask)
    report("block", m(apart, mask), want, atol=REL * float(want.abs().max()))


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("n", [1, 33, 97, 150])  # a work-group's only tile, and rows on their way through LDS beside the next tile's
def test_result_rows(n, c, inplace):
    """Output passes, with the residual (blocks) and without it (a module's update alone)."""
    lib()
    heads = 4
    p = orc.make_block_params(8604, c, c, c // heads, heads)
    m = of3pair.PairStack(c, c, c // heads, heads)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).eval()
    z = orc.make_pair_input(8605, (1,), n, c)
    mask = torch.rand(1, n, n, generator=torch.Generator().manual_seed(8606)) > 0.2
    mask[..., 0] = True  # in 64 bits -1e9 does not absorb the logits of a row without a real key
    mask = mask.float()
    p64 = {k: v.double() for k, v in p.items()}
    print("rows", n, c, inplace, flush=True)
    want = orc.pair_stack_block(z.double(), mask.double(), p64, heads)
    got = m(z.to(DEV), mask.to(DEV), inplace_safe=inplace).cpu()
    report("block", got, want, atol=2 * REL * float(want.abs().max()))
    if not inplace:
        for module, prefix, oracle in ((m.tri_mul_in, "tri_mul_in.", lambda x, k, q: orc.trimul_update(x, k, q, False)),
                                       (m.tri_att_start, "tri_att_start.", lambda x, k, q: orc.triattn_update(x, k, q, heads))):
            q = {k[len(prefix):]: v for k, v in p64.items() if k.startswith(prefix)}
            want = oracle(z.double(), mask.double(), q)
            report(prefix, module(z.to(DEV), mask.to(DEV)).cpu(), want, atol=2 * REL * float(want.abs().max()))


@pytest.mark.parametrize("view", ["flat", "rows"])
@pytest.mark.parametrize("c,n_mult,n", [(64, 2, 1), (64, 2, 31), (64, 2, 129), (64, 2, 187), (128, 4, 182), (128, 4, 183)])
def test_transition_work_groups_of_four_waves(c, n_mult, n, view):
    """One tile, a few and several per work-group; rows that follow one another and rows with a gap (ragged tiles at
    their ends, and at 128 channels an odd number of 32-position tiles in pairs: 183 rows of 6)."""
    lib()
    gen = torch.Generator().manual_seed(8610 + n)
    z = orc.make_pair_input(8611, (1,), n, c)
    mask = (torch.rand(1, n, n, generator=gen) > 0.2).float()
    p = orc.make_transition_params(gen, c, n_mult)
    m = of3pair.SwiGLUTransition(c, n_mult)
    m.load_state_dict(p, strict=True)
    x = z.to(DEV)
    if view == "rows":
        x = torch.zeros(1, n, n + 3, c, device=DEV)[:, :, :n]
        x.copy_(z)
    print("transition", c, n_mult, n, view, flush=True)
    want = orc.transition_update(z.double(), mask.double(), {k: v.double() for k, v in p.items()})
    got = m.to(DEV).eval()(x, mask.to(DEV)).cpu()
    report("update", got, want, atol=REL * float(want.abs().max()))
