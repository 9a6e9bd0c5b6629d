"""What is kept of a block for its later calls does not keep the block."""
import gc
import weakref

import pytest
import torch

import of3pair
from of3pair import _block, pair_stack

PAIRFORMER = (lambda: of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4),
              lambda q, m: _block._pairformer_params(q, m, pair_stack.PairBlock))
CASES = {"pairformer": PAIRFORMER, "pair stack": (lambda: of3pair.PairStack(128, 128, 32, 4), _block._pair_params),
         "template": (lambda: of3pair.TemplatePairBlock(64, 16, 64, 4, fuse_projection_weights=True), _block._pair_params)}


@pytest.mark.parametrize("refused", [False, True])
@pytest.mark.parametrize("case", sorted(CASES))
def test_a_block_goes_with_its_plan(case, refused):
    make, params = CASES[case]
    block = make().eval()
    if refused:
        (block.pair_stack if case == "pairformer" else block).tri_att_end.mha.linear_v = torch.nn.Identity()
    for _ in range(2):
        found = _block._gather(block, lambda q: params(q, block), torch.float32)
        assert (found is None) == refused
    plan = weakref.ref(_block._plans[block][0])
    held, parameter = weakref.ref(block), weakref.ref(next(block.parameters()))
    del block, found
    gc.collect()
    assert held() is None and parameter() is None and plan() is None
