"""The bf16 contraction's tiles of 64 x 64, from 193 tokens on of 64 x 128 (contract_short_kernel): one to eight panels (fewer than its ring holds, as many, more), tiles that
are full, hold one 32 x 32 part in use, or leave waves without any.  The transposed form: test_gpu_pair_join.py, against this one.
Beside them the tiles of 256 x 128 and 256 x 256 at 193 to 256 tokens, which more planes than CUs take there."""
import pytest
import torch

import test_gpu_stages as stages
from gpu_util import bf, lib, report, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [2, 3])
@pytest.mark.parametrize("n", [1, 33, 64, 65, 97, 128, 161, 192, 193, 225, 256])
def test_short(variant, n):
    stages.test_contract_ragged_n(variant, n)


@pytest.mark.parametrize("variant", [2, 3])
@pytest.mark.parametrize("n", [193, 225, 256])
@pytest.mark.parametrize("batch", [2, 3, 5])
def test_many_planes(variant, n, batch):
    """Against fp32 products: one rounding to bf16 (2^-9 of the value, doubled) beside two fp32 sums of kk products in different
    orders (each within kk 2^-24 of the sum of magnitudes, which is below kk).  320 planes take the large tiles (several of them per persistent
    work-group) on any device of at most 319 CUs, 128 and 192 the small ones from 256 CUs on.  Panels past the end are never read (NaN)."""
    L = lib()
    gen = torch.Generator(device="cuda").manual_seed(n + variant + batch)
    CH = 64
    np_, kk = L.of3_padded_n(n), (n + 31) // 32 * 32
    a, b = (bf(torch.randn(batch * CH, np_, np_, generator=gen, device="cuda")) for _ in range(2))
    a[:, :, kk:] = float("nan")
    b[:, :, kk:] = float("nan")
    x = torch.full_like(a, float("nan"))
    print("contract, planes", batch * CH, "variant", variant, "n", n, flush=True)
    ap, bp = stages._to_panels(a), stages._to_panels(b)
    st = L.of3_trimul_contract(ap.data_ptr(), bp.data_ptr(), x.data_ptr(), batch, n, CH, variant, stream())
    assert st == 0, L.of3_status_string(st)
    torch.cuda.synchronize()
    want = torch.bmm(a[:, :, :kk].float(), b[:, :, :kk].float().transpose(1, 2).contiguous())
    report("contract, many planes", x[:, :n, :n], want[:, :n, :n], atol=kk * kk * 2.0 ** -23, rtol=2.0 ** -8)
