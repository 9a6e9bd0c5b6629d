"""The native look at a block's parameters (csrc/host_params.cpp) says what the one in Python says, and leaves to Python what
only Python can answer."""
import os
import sys
from array import array

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openfold-3_amd"))

import of3pair  # noqa: E402
from of3pair import _block  # noqa: E402
from of3pair.pair_stack import PairBlock  # noqa: E402

pytestmark = pytest.mark.skipif(_block._scan is None, reason="host extension not built")


def _gather(block, dtype):
    found = _block._gather(block, lambda q: _block._pairformer_params(q, block, PairBlock), dtype)
    return None if found is None else list(found[0])


def _both(monkeypatch, block, dtype=torch.float32):
    native = _gather(block, dtype)
    again = _gather(block, dtype)
    with monkeypatch.context() as mp:
        mp.setattr(_block, "_scan", None)
        assert _gather(block, dtype) == native == again
    assert _gather(block, dtype) == native
    return native


def test_same_answers(monkeypatch):
    block = of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4).eval()
    first = _both(monkeypatch, block)
    assert first is not None
    lin = block.pair_stack.tri_att_end.mha.linear_v
    keep = lin.weight
    lin.weight = torch.nn.Parameter(keep.detach().clone())  # elsewhere
    moved = _both(monkeypatch, block)
    assert sum(a != b for a, b in zip(first, moved)) == 1
    for other in (keep.detach().to(torch.bfloat16), keep.detach()[:, :64], keep.detach().t()[:, :-1].t(), keep.detach().clone().t()):
        lin.weight = torch.nn.Parameter(other)  # another type, size, layout
        assert (_both(monkeypatch, block) is None) == (not other.is_contiguous() or other.shape != keep.shape or other.dtype != keep.dtype)
    lin.weight = keep
    assert _both(monkeypatch, block) == first
    assert _both(monkeypatch, block, torch.bfloat16) is None
    block.to(torch.bfloat16)
    assert _both(monkeypatch, block, torch.bfloat16) is not None and _both(monkeypatch, block) is None


def test_left_to_python(monkeypatch):
    """A tensor subclass answers for itself; so does a tensor without an address."""

    class Own(torch.Tensor):
        pass

    owner, names, counts = {"a": torch.zeros(4), "b": None}, ["a", "b", "c"], array("q", [4, 1, 1])
    pointers = _block._scan([owner] * 3, names, counts, torch.float32, b"")
    assert array("Q", pointers).tolist() == [owner["a"].data_ptr(), 0, 0]
    assert _block._scan([owner] * 3, names, counts, torch.float32, pointers) is True
    assert _block._scan([owner] * 3, names, counts, torch.float64, pointers) is False
    for odd in (torch.zeros(4).as_subclass(Own), torch.zeros(4).to_sparse(), object()):
        owner["a"] = odd
        assert _block._scan([owner] * 3, names, counts, torch.float32, pointers) is None
    with pytest.raises(ValueError):
        _block._scan([owner], names, counts, torch.float32, b"")
    with pytest.raises(TypeError):
        _block._scan([owner], ["a"], counts, "float32", b"")
