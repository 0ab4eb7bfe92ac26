"""The head's C entry: LN_out scratch in place of its input."""
import pytest
import torch

from krunch_amd import _lib, cpp_path, synthetic

pytestmark = pytest.mark.gpu


def _head(P, x, xn, ld):
    out = torch.full((x.shape[0], ld), 7.0, dtype=torch.float16, device="cuda")
    _lib.call("kr_head_logits", P.ptr, x.data_ptr(), x.shape[0], xn.data_ptr(), out.data_ptr(), ld,
              _lib.stream_ptr())
    return out


# whole 16-row blocks (which the fragment-packed heads take) and not, on both
# sides of the decode head's 512 rows
@pytest.mark.parametrize("M", [5, 16, 256, 512, 513, 528, 1024])
def test_head_in_place(M):
    w = synthetic.make_weights(n_layer=1, C=256, F=256, V=1003, seed=M)
    P = cpp_path.init_weights(w, "cuda")["prepared"]
    try:
        x = torch.randn((M, 256), generator=torch.Generator().manual_seed(M)).half().cuda()
        ref = _head(P, x, torch.empty_like(x), 1005)
        y = x.clone()
        assert torch.equal(_head(P, y, y, 1005), ref)
    finally:
        cpp_path.release_weights(w)
