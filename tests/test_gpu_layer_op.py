"""The layer op's weight copies (transposed and fragment-packed, kept per
weight tensor): how they are made, and calls inside a stream capture."""
import pytest
import torch

from krunch_amd import _lib
from krunch_amd import krunch_ac_hip as ops

pytestmark = pytest.mark.gpu
C, F = 256, 512
SHAPES = ((C, C), (C, C), (C, C), (C, C), (C, F), (F, C), (C, C))


def _inputs(B, T, seed):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g)
    return {"x": rnd(B, T, C).half().cuda(), "ln": [rnd(C).half().cuda() for _ in range(4)],
            "tm": [torch.rand(C, generator=g).half().cuda() for _ in range(5)],
            "decay": (-torch.rand(C, generator=g)).cuda(), "first": torch.zeros(C).cuda(),
            "mats": [(0.05 * rnd(k, n)).half().cuda() for k, n in SHAPES]}


def _state(B):
    h = lambda: torch.zeros(B, C, dtype=torch.float16, device="cuda")
    return [h(), *(torch.zeros(B, C, device="cuda") for _ in range(3)), h()]


def _call(d, st, mats=None):
    m = mats or d["mats"]
    return ops.rwkv4_layer_step_cpp(d["x"], *st, *d["ln"][:2], *d["tm"][:3], d["decay"], d["first"],
                                    *m[:4], *d["ln"][2:], *d["tm"][3:], *m[4:])


# weights never seen before, and weights whose transposed copies det_matmul
# made; a stepped call, a small and a mid-sized window
@pytest.mark.parametrize("warm", [False, True])
@pytest.mark.parametrize("B,T", [(3, 1), (2, 40), (2, 300)])
def test_layer_captured_on_new_weights(B, T, warm):
    """Copies made while a stream is capturing are written when the graph
    runs, so they must not serve a call made before that."""
    d = _inputs(B, T, 10 * B + T)
    ref_st = _state(B)
    ref = _call(d, ref_st, [m.clone() for m in d["mats"]])
    if warm:
        for m in d["mats"]:
            ops.det_matmul(torch.zeros(1, m.shape[0], dtype=torch.float16, device="cuda"), m)
    st = _state(B)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = _call(d, st)
    eager_st = _state(B)
    assert torch.equal(_call(d, eager_st), ref)
    for a, b in zip(eager_st, ref_st):
        assert torch.equal(a, b)
    for _ in range(3):
        for a, b in zip(st, _state(B)):
            a.copy_(b)
        graph.replay()
        assert torch.equal(out, ref)
        for a, b in zip(st, ref_st):
            assert torch.equal(a, b)
        assert torch.equal(_call(d, _state(B)), ref)


# whole and partial tiles of 32 and blocks of 16 columns, one k block and
# several, strides past the row ends
@pytest.mark.parametrize("K,N,ldw,ldt", [(32, 1, 1, 32), (64, 15, 15, 64), (96, 16, 20, 96), (256, 17, 17, 264),
                                         (32, 33, 40, 32), (768, 3072, 3072, 768)])
def test_transpose_pack_equals_the_two_calls(K, N, ldw, ldt):
    W = torch.randn(K, ldw, generator=torch.Generator().manual_seed(K + N)).half().cuda()
    s = _lib.stream_ptr()
    n = _lib.lib().kr_fragment_bytes(N, K) // 2
    wt, ref = (torch.full((N, ldt), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    wf, ref_f = (torch.full((n,), 7.0, dtype=torch.float16, device="cuda") for _ in range(2))
    _lib.call("kr_transpose_pack_f16", W.data_ptr(), ldw, K, N, wt.data_ptr(), ldt, wf.data_ptr(), s)
    _lib.call("kr_transpose_f16", W.data_ptr(), ldw, K, N, ref.data_ptr(), ldt, s)
    _lib.call("kr_pack_fragments", ref.data_ptr(), ldt, N, K, ref_f.data_ptr(), s)
    assert torch.equal(wt, ref) and torch.equal(wf, ref_f)
