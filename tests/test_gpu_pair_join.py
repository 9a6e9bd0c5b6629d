"""A block's call at the lengths where the end of one triangle module and the start of the next are one launch
(pair_join_bf16.hip): the bits of the modules by themselves, for every number of rows per tile, ragged panels and row groups,
batches, the attention before the multiplications, in place and on a transposed tensor."""
import pytest
import torch

import test_gpu_block_call as blocks
import test_gpu_pass_bf16 as passes
from gpu_util import lib  # noqa: F401

import of3pair

pytestmark = pytest.mark.gpu


# (256 CUs) 128 channels: 1 to 6 rows per tile, the first length beyond; 64: 1 to 6 rows, four rows in two and three rounds, beyond
@pytest.mark.parametrize("c,d,n,batch", [(128, 32, 87, 1), (128, 32, 100, 1), (128, 32, 129, 1), (128, 32, 150, 1), (128, 32, 161, 1),
                                         (128, 32, 187, 1), (128, 32, 216, 1), (128, 32, 221, 1), (128, 32, 50, 7),
                                         (64, 16, 100, 2), (64, 16, 129, 1), (64, 16, 161, 2), (64, 16, 187, 2), (64, 16, 205, 2),
                                         (64, 16, 221, 3), (64, 16, 187, 4), (64, 16, 256, 1), (64, 16, 256, 4), (64, 16, 257, 1)])
def test_joined(monkeypatch, c, d, n, batch):
    passes.test_shared_pass(monkeypatch, c, d, n, batch, True)


@pytest.mark.parametrize("n,batch", [(1, 1), (33, 2), (100, 2), (187, 2), (221, 3)])
def test_attention_first(monkeypatch, n, batch):
    lib()
    m = blocks._fill(of3pair.TemplatePairBlock(64, 16, 64, 4, tri_mul_first=False), n).to("cuda").to(torch.bfloat16).eval()
    gen = torch.Generator().manual_seed(n)
    t = torch.randn(batch, n, n, 64, generator=gen).to("cuda").to(torch.bfloat16)
    mask = (torch.rand(batch, n, n, generator=gen) > 0.2).float().to("cuda")
    want = blocks._by_modules(monkeypatch, lambda: m(t, mask))
    assert torch.isfinite(want.float()).all()
    assert torch.equal(m(t, mask), want)
