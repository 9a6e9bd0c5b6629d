"""What kernels would read outside their memory is refused before a launch: parameters and masks that live elsewhere than the
activations, parameters of other sizes than the activations' channels."""
import os
import sys
from array import array

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "openfold-3_amd"))

import of3pair  # noqa: E402
from of3pair import _block  # noqa: E402
from of3pair import functional as F3  # noqa: E402
from of3pair.pair_stack import PairBlock  # noqa: E402

ELSEWHERE = torch.device("cuda", 0)  # a device object needs no GPU


def test_masks_and_parameters_elsewhere():
    with pytest.raises(RuntimeError, match="must live on cuda:0"):
        F3._mask_arg(torch.ones(1, 4, 4), (1,), 1, 4, ELSEWHERE)
    assert F3._mask_arg(torch.ones(1, 4, 4), (1,), 1, 4, torch.device("cpu"))[0] is not None

    class OnTheGpu:  # stands for the activations
        device, dtype, shape = ELSEWHERE, torch.float32, (1, 4, 4, 8)

    with pytest.raises(RuntimeError, match="must live on cuda:0"):
        F3._w(torch.zeros(8), OnTheGpu, 8)


def test_parameter_sizes():
    x = torch.zeros(1, 4, 4, 8)
    assert F3._w(torch.zeros(8), x, 8).numel() == 8
    for other in (torch.zeros(7), torch.zeros(16), torch.zeros(8, 8)):
        with pytest.raises(ValueError, match="does not fit"):
            F3._w(other, x, 8)


@pytest.mark.parametrize("native", [True, False])
def test_a_block_elsewhere_is_not_gathered(monkeypatch, native):
    if native and _block._scan is None:
        pytest.skip("host extension not built")
    if not native:
        monkeypatch.setattr(_block, "_scan", None)
    block = of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4).eval()

    def gather(device):
        return _block._gather(block, lambda q: _block._pairformer_params(q, block, PairBlock), torch.float32, device)

    for _ in range(2):  # the first time and where the pointers are those of the call before
        assert gather(None) is not None and gather(torch.device("cpu")) is not None
        assert gather(ELSEWHERE) is None
    if native:
        owner, counts = {"a": torch.zeros(4)}, array("q", [4])
        assert _block._scan([owner], ["a"], counts, torch.float32, b"", 0) is False
        assert isinstance(_block._scan([owner], ["a"], counts, torch.float32, b"", -1), bytes)
        with pytest.raises(TypeError):
            _block._scan([owner], ["a"], counts, torch.float32, b"", None)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("by_modules", [False, True])
def test_refused_by_the_modules(monkeypatch, dtype, by_modules):
    """Through the public entry points.  Every refusal comes from the host before the first launch that would read there."""
    torch.manual_seed(0)
    n = 40
    block = of3pair.PairFormerBlock(384, 128, 24, 16, 128, 32, 4).to("cuda").to(dtype).eval()
    s, z = torch.randn(1, n, 384, device="cuda", dtype=dtype), torch.randn(1, n, n, 128, device="cuda", dtype=dtype)
    single, pair = torch.ones(1, n, device="cuda"), torch.ones(1, n, n, device="cuda")
    if by_modules:
        monkeypatch.setattr(_block, "_gather", lambda *args: None)
    for _ in range(2):
        want = block(s, z, single, pair)
    for masks in ((single, pair.cpu()), (single.cpu(), pair)):
        with pytest.raises(RuntimeError, match="mask must live on cuda"):
            block(s, z, *masks)
    for part, name in ((block.pair_stack.tri_att_end.mha.linear_v, "weight"), (block.pair_stack.tri_mul_out.layer_norm_in, "bias"),
                       (block.single_transition.linear_out, "weight"), (block.attn_pair_bias.linear_z, "weight")):
        keep = getattr(part, name)
        setattr(part, name, torch.nn.Parameter(keep.detach().cpu()))
        with pytest.raises(RuntimeError, match="parameter must live on cuda"):
            block(s, z, single, pair)
        setattr(part, name, keep)
    for narrow in (of3pair.TriangleMultiplicationOutgoing(64, 64), of3pair.TriangleAttention(64, 16, 4), of3pair.SwiGLUTransition(64, 2),
                   of3pair.PairStack(64, 64, 16, 4)):
        with pytest.raises(ValueError):
            narrow.to("cuda").to(dtype).eval()(z, pair)
    got = block(s, z, single, pair)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
