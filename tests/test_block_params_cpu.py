"""Which blocks the single call takes (of3pair._block): the choice reads parameters and modules only, no device."""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openfold-3_amd"))

import of3pair  # noqa: E402
from of3pair import _block  # noqa: E402
from of3pair.pair_stack import PairBlock  # noqa: E402


def _taken(block):
    return _block._gather(block, lambda q: _block._pairformer_params(q, block, PairBlock), torch.float32) is not None


def test_forward_of_a_submodules_own():
    """A forward set on an instance (as wrappers that move weights between devices do) is what the block has to call."""
    block = of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4).eval()
    assert _taken(block)
    for sub in (block.single_transition, block.attn_pair_bias, block.pair_stack, block.pair_stack.pair_transition):
        sub.forward = sub.forward
        assert not _taken(block)
        del sub.forward
        assert _taken(block)


def test_first_call_of_a_long_sequence():
    """Starts module by module, once; shorter ones do not, and a tensor that no module takes is left to them."""
    block = of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4).eval()
    n = _block._LATE_FROM
    assert not _block._first_call(block, torch.empty(n - 1, n - 1, 1, device="meta"))
    assert not _block._first_call(block, torch.empty(n))
    assert _block._first_call(block, torch.empty(1, n, n, 1, device="meta"))
    assert not _block._first_call(block, torch.empty(1, n, n, 1, device="meta"))
    assert _taken(block)


def test_smaller_parameter_at_the_same_address():
    """What is kept between calls is the pointers: a parameter replaced by a part of itself has to be seen."""
    block = of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4).eval()
    assert _taken(block)
    for sub in (block.pair_stack.tri_mul_in.linear_z, block.pair_stack.tri_att_end.layer_norm, block.single_transition.linear_out,
                block.attn_pair_bias.mha.linear_q):
        whole = sub.weight
        sub.weight = torch.nn.Parameter(whole.data[: whole.shape[0] // 2])
        assert sub.weight.data_ptr() == whole.data_ptr() and not _taken(block)
        sub.weight = whole
        assert _taken(block)
