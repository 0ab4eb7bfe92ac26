"""Packed WKV: the time-split kernel (32-token chunks, 16-channel slices)
against the recurrence run token by token, bit for bit, and against the fp32
oracle."""
import numpy as np
import pytest
import torch

from krunch_amd import _lib, cpp_path, synthetic
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


# the last workgroup count that takes the time-split kernel and the first that
# does not, at one to two chunks and above, per codec; T short of and past a chunk
@pytest.mark.parametrize("w8a8,B,T", [(False, 64, 33), (False, 65, 33), (False, 96, 65), (False, 97, 65),
                                      (True, 128, 40), (True, 129, 40), (True, 160, 64), (True, 161, 64)])
def test_layers_on_both_sides_of_the_split_line(w8a8, B, T):
    """Packed layers whose WKV changes kernels against the same tokens one
    stream at a time (always the time-split kernel): equal bit for bit."""
    w = synthetic.make_weights(n_layer=2, C=256, F=512, V=300, seed=3)
    W = cpp_path.init_weights(w, "cuda", w8a8=w8a8)
    try:
        ids = torch.from_numpy(synthetic.zipf_tokens(B, T, V=300))
        st = cpp_path.fresh_state_batched(W, B)
        got = cpp_path.forward_packed_batched(W, ids, st).view(B, T, -1)
        for b in (0, B // 2, B - 1):
            st1 = cpp_path.fresh_state_batched(W, 1)
            assert torch.equal(cpp_path.forward_packed_batched(W, ids[b:b + 1], st1), got[b]), b
            for x, y in zip(st1.flat(), st.flat()):
                assert torch.equal(x[0], y[b]), b
    finally:
        cpp_path.release_weights(w)
