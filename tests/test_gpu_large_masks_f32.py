"""fp32 triangle multiplication on two fp16 terms: masks of any finite size.  a and b carry the mask, whose largest value the
launch that splits the weights takes; plain fp32's own error is the bound, as in test_gpu_uneven_parameters_f32."""
import pytest
import torch

from gpu_util import lib, report  # noqa: F401
from oracle import pairstack_oracle as orc
from test_gpu_uneven_parameters_f32 import DEV, _check

import of3pair

pytestmark = pytest.mark.gpu

MASKS = {
    "0 to 1000": lambda gen, n: torch.tensor([0.0, 0.25, 1.0, 300.0, 1000.0])[torch.randint(0, 5, (1, n, n), generator=gen)],
    "256": lambda gen, n: torch.full((1, n, n), 256.0),
    "3e4 beside 1": lambda gen, n: torch.where(torch.rand(1, n, n, generator=gen) > 0.98, 3e4, 1.0),
    "-1e6": lambda gen, n: -1e6 * torch.rand(1, n, n, generator=gen),
    "1e-9": lambda gen, n: 1e-9 * torch.rand(1, n, n, generator=gen),
    "zeros": lambda gen, n: torch.zeros(1, n, n),
    "last": lambda gen, n: torch.ones(1, n, n).index_put((torch.tensor([0]), torch.tensor([n - 1]), torch.tensor([n - 1])), torch.tensor(700.0)),
}


@pytest.mark.parametrize("c", [64, 128])
@pytest.mark.parametrize("n", [5, 33, 90, 300])
@pytest.mark.parametrize("what", MASKS)
def test_trimul_masks(what, n, c):
    lib()
    gen = torch.Generator().manual_seed(8900 + n)
    p = orc.make_trimul_params(gen, c, c)
    # Beside a value 2^r times as large one of 1 loses what its 22 bits have below 2^-37+r of its bound: 0 up to some 2^10, 1e-6 at 3e4
    spread = 2.0**-34 * 3e4 if what.startswith("3e4") else 0.0
    z, mask = orc.make_pair_input(8901, (1,), n, c), MASKS[what](gen, n)
    print("mask", what, n, c, flush=True)
    for cls, outgoing in ((of3pair.TriangleMultiplicationOutgoing, True), (of3pair.TriangleMultiplicationIncoming, False)):
        _check("mask %s, %d, %d" % (what, n, c), cls(c, c), [z, mask], lambda x, m, q: orc.trimul_update(x, m, q, outgoing), p,
               spread)


@pytest.mark.parametrize("view", ["plain", "transposed", "one row", "batch", "off 16 bytes"])
def test_trimul_mask_views(view):
    lib()
    c, n, b = 128, 37, 3
    gen = torch.Generator().manual_seed(8910)
    p = orc.make_trimul_params(gen, c, c)
    m = of3pair.TriangleMultiplicationOutgoing(c, c)
    m.load_state_dict(p, strict=True)
    z = orc.make_pair_input(8911, (b,), n, c)
    mask = 1000.0 * torch.rand(b, n, n, generator=gen)
    mask[b - 1, n - 1, n - 1] = 5e5  # the last value of all
    if view == "transposed":
        mask = mask.to(DEV).transpose(-1, -2)
    elif view == "one row":
        mask = mask[:, n - 1:].to(DEV).expand(b, n, n)
    elif view == "plain":
        mask = mask.to(DEV)
    elif view == "off 16 bytes":
        mask = torch.empty(mask.numel() + 1, device=DEV)[1:].view(mask.shape).copy_(mask)
    else:
        mask = mask[b - 1:].to(DEV).expand(b, n, n)
    print("mask view", view, flush=True)
    want = orc.trimul_update(z.double(), mask.cpu().double(), {k: v.double() for k, v in p.items()}, True)
    got = m.to(DEV).eval()(z.to(DEV), mask).cpu()
    report("update", got, want, atol=1e-5 * float(want.abs().max()))


def test_one_large_value():
    """Wherever it lies: a value left out of the maximum would make a or b infinite (64 work-groups take 524288 values a round)."""
    lib()
    c, n = 64, 740
    gen = torch.Generator().manual_seed(8915)
    m = of3pair.TriangleMultiplicationOutgoing(c, c)
    m.load_state_dict(orc.make_trimul_params(gen, c, c), strict=True)
    m = m.to(DEV).eval()
    z = orc.make_pair_input(8916, (1,), n, c).to(DEV)
    for at in (0, 3, 1023, 65535, 131072, 262143, 524287, 524288, 540000, n * n - 4, n * n - 1):
        mask = torch.ones(1, n, n, device=DEV)
        mask.view(-1)[at] = 1e6
        print("large value at", at, flush=True)
        assert m(z, mask).isfinite().all() and m(z, mask.transpose(-1, -2)).isfinite().all()


def test_value_that_is_no_number():
    """It makes its own row and column no numbers and leaves the others as they were."""
    lib()
    c, n = 64, 40
    gen = torch.Generator().manual_seed(8920)
    p = orc.make_trimul_params(gen, c, c)
    m = of3pair.TriangleMultiplicationOutgoing(c, c)
    m.load_state_dict(p, strict=True)
    m = m.to(DEV).eval()
    z = orc.make_pair_input(8921, (1,), n, c).to(DEV)
    mask = (torch.rand(1, n, n, generator=gen) > 0.2).float().to(DEV)
    want = m(z, mask)
    for value in (float("nan"), float("inf")):
        mask[0, 7, 9] = value
        got = m(z, mask)
        rest = torch.arange(n, device=DEV) != 7
        assert got[:, 7].isnan().all() and got[:, :, 7].isnan().all()
        assert torch.equal(got[:, rest][:, :, rest], want[:, rest][:, :, rest])


def _fill(module, gen):
    with torch.no_grad():
        for name, p in module.named_parameters():
            r = torch.randn(p.shape, generator=gen)
            p.copy_(r / p.shape[1] ** 0.5 if p.dim() == 2 else (1.0 if name.endswith("weight") else 0.0) + 0.1 * r)
    return module.to(DEV).eval()


def _mask(n):
    mask = torch.full((1, n, n), 1000.0, device=DEV)
    mask[..., 5] = 3.0
    return mask


@pytest.mark.parametrize("c", [64, 128])
def test_block_masks(c):
    """Through the call of a whole block, whose weights are split together, against the modules one by one."""
    lib()
    n = 41
    gen = torch.Generator().manual_seed(8930)
    m = _fill(of3pair.PairStack(c, c, c // 4, 4), gen)
    z = orc.make_pair_input(8931, (1,), n, c).to(DEV)
    print("block mask", c, flush=True)
    want = m._modules_forward(z, _mask(n), False, False)
    assert want.isfinite().all()
    report("block", m(z, _mask(n)), want, atol=1e-5 * float(want.abs().max()))


def test_stack_masks():
    """Blocks whose weights are split four at a time, against blocks one by one."""
    lib()
    n = 41
    stack = _fill(of3pair.PairFormerStack(384, 128, 24, 16, 128, 32, 4, no_blocks=6, transition_n=4), torch.Generator().manual_seed(8940))
    s = torch.randn(1, n, 384, generator=torch.Generator().manual_seed(8941)).to(DEV)
    z = orc.make_pair_input(8942, (1,), n, 128).to(DEV)
    single = torch.ones(1, n, device=DEV)
    print("stack mask", flush=True)
    with torch.no_grad():
        got = stack(s, z, single, _mask(n))
        want = s, z
        for block in stack.blocks:
            want = block(want[0], want[1], single, _mask(n))
    for g, w in zip(got, want):
        assert w.isfinite().all()
        report("stack", g, w, atol=1e-5 * float(w.abs().max()))
