"""Stepped layers with the LN-mix inside the product launches (few streams)
against packed windows over the same tokens, and the decode run's refusal of a
stream under capture."""
import ctypes

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


# layers of four launches and of six, both codecs
@pytest.mark.parametrize("w8a8", [False, True])
@pytest.mark.parametrize("B", [1, 5, 100, 200])
def test_step_timing_leaves_the_launches_as_they_are(B, w8a8):
    """A captured decode step has as many launches with a phase timed as
    without; an eager one reports a dispatch and a wave span per layer."""
    w = synthetic.make_weights(n_layer=3, V=1000, seed=B)
    P = cpp_path.init_weights(w, "cuda", w8a8=w8a8)["prepared"]
    dev = dict(device="cuda")
    syms = torch.zeros(B, dtype=torch.int32, **dev)
    bits = torch.zeros(64, dtype=torch.uint8, **dev)
    ac = torch.zeros((B, 4), dtype=torch.uint32, **dev)
    st = cpp_path.fresh_state_batched({"prepared": P}, B)
    x = torch.zeros((B, P.C), dtype=torch.float16, **dev)
    ws = torch.empty(_lib.lib().kr_forward_workspace_bytes(B, P.C, P.F), dtype=torch.uint8, **dev)
    logits = torch.empty((B, P.V), dtype=torch.float16, **dev)
    L = _lib.lib()
    _lib.call("kr_decode_init_batched", bits.data_ptr(), 64, None, None, ac.data_ptr(), B, _lib.stream_ptr())

    def step():
        _lib.call("kr_decode_step", P.ptr, B, st.ptr, syms.data_ptr(), x.data_ptr(), ws.data_ptr(),
                  ws.numel(), logits.data_ptr(), P.V, bits.data_ptr(), 64, None, None, ac.data_ptr(),
                  None, 0, None, None, 24, _lib.stream_ptr())

    def launches():
        g = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(g):
            step()
        n = ctypes.c_size_t(0)
        assert L.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
        return n.value

    try:
        step()
        plain = launches()
        for phase in (3, 5, 6):
            _lib.call("kr_step_timing", phase, None)
            assert launches() == plain, phase
            step()
            us, span, n = (ctypes.c_double * 8)(), (ctypes.c_double * 8)(), ctypes.c_int(0)
            _lib.call("kr_step_timing_read", us, span, 8, ctypes.byref(n))
            assert n.value == 3
            assert all(0.0 < us[i] < 1000.0 and 0.0 < span[i] < 1000.0 for i in range(3)), phase
    finally:
        L.kr_step_timing(-1, None)
        cpp_path.release_weights(w)


# the last row counts of four launches per layer and the first of six, at the
# widths and codecs whose lines are not among the sizes above; at C = 512, 129
# rows are also the first with two column panels in the O and V products
@pytest.mark.parametrize("C,w8a8,Bs", [(256, False, (160, 161)), (256, True, (12, 13, 96, 97, 128, 129)),
                                       (512, False, (128, 129, 160, 161)), (512, True, (128, 129)),
                                       (1024, False, (48, 49)), (1024, True, (96, 97))])
def test_stepped_equals_packed_at_the_lines(C, w8a8, Bs):
    test_stepped_equals_packed(C, Bs, w8a8)


def test_decode_run_refuses_a_capturing_stream():
    """With use_graph the run waits for its steps on the caller's stream; on
    one that is being captured it is an error, and the capture goes on."""
    w = synthetic.make_weights(n_layer=2, V=300, seed=4)
    P = cpp_path.init_weights(w, "cuda")["prepared"]
    B, dev = 3, dict(device="cuda")
    syms = torch.full((B,), 5, dtype=torch.int32, **dev)
    bits = torch.zeros(64, dtype=torch.uint8, **dev)
    ac = torch.zeros((B, 4), dtype=torch.uint32, **dev)
    st = cpp_path.fresh_state_batched({"prepared": P}, B)
    x = torch.zeros((B, P.C), dtype=torch.float16, **dev)
    ws = torch.empty(_lib.lib().kr_decode_workspace_bytes(B, 1, P.C, P.F), dtype=torch.uint8, **dev)
    logits = torch.empty((B, P.V), dtype=torch.float16, **dev)
    before = st.buf.clone()
    y = torch.zeros(4, **dev)
    torch.cuda.synchronize()

    def run():
        _lib.call("kr_decode_run", P.ptr, B, st.ptr, syms.data_ptr(), x.data_ptr(), ws.data_ptr(),
                  ws.numel(), logits.data_ptr(), P.V, bits.data_ptr(), 64, None, None, ac.data_ptr(),
                  None, 0, None, None, 24, 2, 1, 1, _lib.stream_ptr())

    try:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y.add_(1.0)
            with pytest.raises(_lib.KrunchError, match="captured"):
                run()
            y.add_(1.0)
        for i in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert y.tolist() == [2.0 * (i + 1)] * 4
        assert torch.equal(st.buf, before) and syms.tolist() == [5] * B
    finally:
        cpp_path.release_weights(w)
