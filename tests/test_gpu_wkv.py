"""Packed WKV: the time-split kernel (32-token chunks, 16-channel slices)
against the recurrence run token by token, bit for bit, and against the fp32
oracle."""
import numpy as np
import pytest
import torch

from krunch_amd import _lib
from oracle import rwkv4

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _wkv(k, v, r, w, u, state):
    B, T, C = k.shape
    ry = torch.empty((B, T, C), dtype=torch.float16, device=DEV)
    _lib.call("kr_wkv", B, T, C, w.data_ptr(), u.data_ptr(), k.data_ptr(), v.data_ptr(),
              r.data_ptr(), *(s.data_ptr() for s in state), ry.data_ptr(), _lib.stream_ptr())
    return ry


# one token short of, at and past one and two chunks; a channel count that is
# no multiple of 16; the widest; enough streams for the sequential kernel
@pytest.mark.parametrize("B,T,C", [(2, 31, 768), (2, 32, 768), (1, 33, 100), (3, 63, 17), (2, 64, 1024),
                                   (1, 65, 256), (1, 200, 768), (40, 40, 768)])
def test_packed_wkv_equals_token_by_token(B, T, C):
    g = torch.Generator().manual_seed(B * 1000 + T + C)
    k = (1.5 * torch.randn(B, T, C, generator=g)).to(DEV)
    v = torch.randn(B, T, C, generator=g).to(DEV)
    r = torch.sigmoid(torch.randn(B, T, C, generator=g)).half().to(DEV)
    w = -torch.exp(torch.linspace(-5.0, 3.0, C)).to(DEV)
    u = torch.full((C,), -1.2, device=DEV)
    fresh = lambda: [torch.zeros(B, C, device=DEV), torch.zeros(B, C, device=DEV),
                     torch.full((B, C), -1e30, device=DEV)]
    st, st1 = fresh(), fresh()
    got = _wkv(k, v, r, w, u, st)
    for t in range(T):
        one = _wkv(*(x[:, t:t + 1].contiguous() for x in (k, v, r)), w, u, st1)
        assert torch.equal(one[:, 0], got[:, t]), t
    for a, b in zip(st, st1):
        assert torch.equal(a, b)
    ost = {"aa": torch.zeros(B, C), "bb": torch.zeros(B, C), "pp": torch.full((B, C), -1e30)}
    y = rwkv4.wkv(k.cpu(), v.cpu(), w.cpu(), u.cpu(), ost)
    # y and the product are rounded to fp16 once each (2^-11 relative), on top
    # of exp and reciprocal errors far below that
    ref = (r.float().cpu() * y).numpy()
    np.testing.assert_allclose(got.float().cpu().numpy(), ref, rtol=2.0 ** -9, atol=2.0 ** -9)
