"""Stepped layers with the LN-mix inside the product launches (few streams)
against packed windows over the same tokens, and the decode run's refusal of a
stream under capture."""
import numpy as np
import pytest
import torch

from krunch_amd import _lib, cpp_path, synthetic
from krunch_amd.inference import InferenceEngine

pytestmark = pytest.mark.gpu


# one row per wave and more, the last and first rows of 16-row tiles, each
# split of the waves and panels, the last of each codec's range and the first
# beyond; the other widths at the smallest and largest tile
@pytest.mark.parametrize("w8a8", [False, True])
@pytest.mark.parametrize("C,Bs", [(768, (1, 4, 7, 10, 15, 16, 17, 33, 80, 81, 128, 129, 160, 161)),
                                  (256, (1, 16, 130)), (512, (5, 100)), (1024, (1, 20, 128, 160))])
def test_stepped_equals_packed(C, Bs, w8a8):
    w = synthetic.make_weights(n_layer=2, C=C, F=4 * C, V=1000, seed=C + 1)
    W = cpp_path.init_weights(w, "cuda", w8a8=w8a8)
    try:
        for B in Bs:
            ids = torch.from_numpy(synthetic.zipf_tokens(B, 3, V=1000, seed_base=B))
            st, st2 = (cpp_path.fresh_state_batched(W, B) for _ in range(2))
            packed = cpp_path.forward_packed_batched(W, ids, st).view(B, 3, -1)
            stepped = [cpp_path.forward_stepped_batched(W, ids[:, t], st2) for t in range(3)]
            assert torch.equal(packed, torch.stack(stepped, 1)), B
            assert torch.equal(st.buf, st2.buf), B
    finally:
        cpp_path.release_weights(w)


def test_decode_on_another_stream():
    """The decode graphs run on the caller's stream, whichever it is."""
    e = InferenceEngine().load(synthetic.make_weights(n_layer=2, V=1000))
    toks = list(synthetic.zipf_tokens(5, 40, V=1000))
    enc = e.compress_tokens_batched(toks)
    with torch.cuda.stream(torch.cuda.Stream()):
        assert e.compress_tokens_batched(toks) == enc
        dec = e.decompress_tokens_batched(enc)
    for t, d in zip(toks, dec):
        np.testing.assert_array_equal(d, t)


def test_packed_product_refuses_more_than_512_rows():
    """The fragment-packed product's own entry keeps its row limit."""
    xf = torch.zeros(528 * 256, dtype=torch.float16, device="cuda")
    wf = torch.zeros(256 * 256, dtype=torch.float16, device="cuda")
    out = torch.empty((513, 256), dtype=torch.float16, device="cuda")
    with pytest.raises(Exception, match="512"):
        _lib.call("kr_det_matmul_packed", xf.data_ptr(), 513, 256, wf.data_ptr(), 256, out.data_ptr(),
                  256, 1, None, None, 0, _lib.stream_ptr())
    with pytest.raises(Exception, match="512"):
        _lib.call("kr_det_matmul_i8", xf.data_ptr(), out.data_ptr(), 513, 256, wf.data_ptr(),
                  out.data_ptr(), 256, out.data_ptr(), 256, 1, None, None, 1, _lib.stream_ptr())
