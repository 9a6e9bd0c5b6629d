"""bf16 triangle attention core on logits of several hundreds that the q k products carry: the pass with running maxima, whose
offset has to be that of the finished logits; and rows of masked keys whose logits the mask bias does not take up."""
import math

import pytest
import torch

from gpu_util import bf, lib, report, stream
from test_gpu_stages import DEV, LOG2E, _gen, _randn, _to_panels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("n", [33, 64, 130, 420])
def test_large_logits(D, n):
    L = lib()
    B, H = 1, 4
    gen = _gen(47 * n + D)
    np_ = L.of3_padded_n(n)
    q, k, vt = bf(60.0 * _randn(gen, B, n, H, np_, D)), bf(_randn(gen, B, n, H, np_, D)), bf(_randn(gen, B, n, H, D, np_))
    tb = _randn(gen, B, H, n, np_).contiguous()
    mask = torch.ones(B, n, n, device=DEV)
    mask[:, 3::7, ::3] = 0
    mb = torch.full((B, n, np_), float("-inf"), device=DEV)
    mb[..., :n] = LOG2E * 1e9 * (mask - 1)
    o = torch.full((B, n, n, H * D), float("nan"), dtype=torch.bfloat16, device=DEV)
    print("large logits", D, n, flush=True)
    vtp = _to_panels(vt)
    st = L.of3_triattn_flash(q.data_ptr(), k.data_ptr(), vtp.data_ptr(), tb.data_ptr(), mb.data_ptr(), o.data_ptr(), B, n, H, D,
                             stream())
    assert st == 0, L.of3_status_string(st)
    torch.cuda.synchronize()
    qf, kf, vf = q[:, :, :, :n].float(), k[:, :, :, :n].float(), vt[..., :n].float()
    s = (qf @ kf.transpose(-1, -2).contiguous() + mb[:, :, None, None, :n]) + tb[:, None, :, :, :n]
    p = torch.softmax(s * math.log(2.0), dim=-1)
    want = (p @ vf.transpose(-1, -2).contiguous()).permute(0, 1, 3, 2, 4).reshape(B, n, n, H * D)
    # weights and v are rounded to bf16 as in the other tests of this kernel
    report("flash o (large logits)", o, want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("n", [33, 64, 150, 451])
def test_masked_rows_of_large_logits(D, n):
    """Beside -1.44e9 fp32 values are 128 apart: the keys whose bias rounds to the largest multiple share the weight."""
    L = lib()
    B, H = 1, 4
    gen = _gen(53 * n + D)
    np_ = L.of3_padded_n(n)
    q, k, vt = bf(0.0 * _randn(gen, B, n, H, np_, D)), bf(_randn(gen, B, n, H, np_, D)), bf(_randn(gen, B, n, H, D, np_))
    tb = (128.0 * torch.randint(-6, 7, (B, H, n, np_), generator=torch.Generator().manual_seed(n)).float()).to(DEV)
    mask = torch.ones(B, n, n, device=DEV)
    mask[:, 2:9] = 0
    mb = torch.full((B, n, np_), float("-inf"), device=DEV)
    mb[..., :n] = LOG2E * 1e9 * (mask - 1)
    o = torch.full((B, n, n, H * D), float("nan"), dtype=torch.bfloat16, device=DEV)
    print("masked rows of large logits", D, n, flush=True)
    vtp = _to_panels(vt)
    st = L.of3_triattn_flash(q.data_ptr(), k.data_ptr(), vtp.data_ptr(), tb.data_ptr(), mb.data_ptr(), o.data_ptr(), B, n, H, D,
                             stream())
    assert st == 0, L.of3_status_string(st)
    torch.cuda.synchronize()
    mb16 = mb[..., :n].bfloat16().float()  # as the kernel adds it: a multiple of 128
    s = mb16[:, :, None, None] + tb[:, None, :, :, :n]
    p = torch.softmax((s - s.max(-1, keepdim=True).values) * math.log(2.0), dim=-1)
    want = (p @ vt[..., :n].float().transpose(-1, -2).contiguous()).permute(0, 1, 3, 2, 4)
    # weights and v are rounded to bf16 as in the other tests of this kernel
    report("flash o (masked rows)", o, want.reshape(B, n, n, H * D), atol=2e-2, rtol=2e-2)
