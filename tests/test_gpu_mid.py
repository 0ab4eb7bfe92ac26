"""Packed windows of a few hundred to a few thousand rows (fragment-packed
operands through the register-fed product kernel) against the same tokens in
windows of at most 512 rows, which the small-M kernels run: the reduction
contract makes them equal bit for bit, state included."""
import pytest
import torch

from krunch_amd import _lib, cpp_path, krunch_ac_hip, synthetic

pytestmark = pytest.mark.gpu


# row counts at the first past the small-M kernels, inside and at the edges of
# 48- and 64-row tiles, the last of each codec's range and the first beyond
@pytest.mark.parametrize("w8a8", [False, True])
@pytest.mark.parametrize("B,T", [(1, 513), (3, 213), (1, 768), (7, 143), (1, 1664), (5, 333), (16, 144),
                                 (5, 461)])
def test_mid_window_equals_small_windows(B, T, w8a8):
    w = synthetic.make_weights(n_layer=2, C=768, F=3072, V=1000, seed=5)
    W = cpp_path.init_weights(w, "cuda", w8a8=w8a8)
    try:
        ids = torch.from_numpy(synthetic.zipf_tokens(B, T, V=1000, seed_base=B + T))
        st, st2 = (cpp_path.fresh_state_batched(W, B) for _ in range(2))
        whole = cpp_path.forward_packed_batched(W, ids, st).view(B, T, -1)
        step = 512 // B
        parts = [cpp_path.forward_packed_batched(W, ids[:, i:i + step].contiguous(), st2).view(
            B, -1, whole.shape[-1]) for i in range(0, T, step)]
        assert torch.equal(whole, torch.cat(parts, 1))
        assert torch.equal(st.buf, st2.buf)
    finally:
        cpp_path.release_weights(w)


def test_layer_op_repacks_a_changed_weight():
    """The layer op's packed weight copies follow an in-place change."""
    C, F, B, T = 256, 512, 2, 300
    g = torch.Generator().manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g)
    vec = [rnd(C).half().cuda() for _ in range(5)]
    tm = [torch.rand(C, generator=g).half().cuda() for _ in range(4)]
    mats = [(0.05 * rnd(k, n)).half().cuda() for k, n in
            ((C, C), (C, C), (C, C), (C, C), (C, F), (F, C), (C, C))]
    decay, first = (-torch.rand(C, generator=g)).cuda(), torch.zeros(C).cuda()
    x = rnd(B, T, C).half().cuda()

    def step(m):
        st = [torch.zeros(B, C, dtype=torch.float16, device="cuda"), *(torch.zeros(B, C, device="cuda")
              for _ in range(3)), torch.zeros(B, C, dtype=torch.float16, device="cuda")]
        return krunch_ac_hip.rwkv4_layer_step_cpp(
            x, *st, vec[0], vec[1], tm[0], tm[1], tm[2], decay, first, *m[:4], vec[2], vec[3], tm[3],
            vec[4], *m[4:])

    before = step(mats)
    mats[5].mul_(-1.0)
    after = step(mats)
    assert not torch.equal(before, after)
    assert torch.equal(after, step([m.clone() for m in mats]))


# rows past the decode head's 512, at and around its 256-row groups and
# 16-row blocks; row strides of every alignment; column counts with and
# without a last partial block, fewer blocks than a run's pipeline, and
# widths with 8, 16 and 24 fragments per row
@pytest.mark.parametrize("C,V,M,ld", [(768, 1000, 528, 1000), (768, 1003, 513 + 15, 1003), (768, 50277, 784, 50277),
                                      (768, 1001, 1040, 1002), (512, 777, 2064, 779), (256, 40, 768, 41),
                                      (768, 3, 544, 5), (256, 5000, 8208, 5000), (512, 2000, 512 + 256, 2000)])
def test_head_rows_equals_single_blocks(C, V, M, ld):
    """The head over many rows against the same rows 256 at a time (the decode
    head): the one-chain contract makes them equal bit for bit. Nothing is
    written past a row's V columns."""
    w = synthetic.make_weights(n_layer=1, C=C, F=4 * C, V=V, seed=C + V)
    P = cpp_path.init_weights(w, "cuda")["prepared"]
    try:
        g = torch.Generator(device="cuda").manual_seed(M)
        x = torch.randn((M, C), generator=g, device="cuda").half()
        xn = torch.empty_like(x)
        s = _lib.stream_ptr()
        got = torch.full((M, ld), 7.0, dtype=torch.float16, device="cuda")
        ref = got.clone()
        _lib.call("kr_head_logits", P.ptr, x.data_ptr(), M, xn.data_ptr(), got.data_ptr(), ld, s)
        for r in range(0, M, 256):
            n = min(256, M - r)
            _lib.call("kr_head_logits", P.ptr, x[r:].data_ptr(), n, xn.data_ptr(), ref[r:].data_ptr(), ld, s)
        assert torch.equal(got, ref)
        assert bool((got[:, V:] == 7.0).all())
    finally:
        cpp_path.release_weights(w)


# the last row counts of the register-fed kernel and the first past it, where
# the line lies elsewhere than above
@pytest.mark.parametrize("C,w8a8,B,T", [(768, False, 17, 128), (768, False, 7, 311), (1024, False, 1, 1856),
                                        (1024, False, 3, 619), (1024, True, 3, 512), (1024, True, 29, 53),
                                        (256, False, 9, 256), (256, False, 5, 461)])
def test_windows_on_both_sides_of_the_lines(C, w8a8, B, T):
    w = synthetic.make_weights(n_layer=2, C=C, F=4 * C, V=500, seed=C)
    W = cpp_path.init_weights(w, "cuda", w8a8=w8a8)
    try:
        ids = torch.from_numpy(synthetic.zipf_tokens(B, T, V=500, seed_base=B + T))
        st, st2 = (cpp_path.fresh_state_batched(W, B) for _ in range(2))
        whole = cpp_path.forward_packed_batched(W, ids, st).view(B, T, -1)
        step = 512 // B
        parts = [cpp_path.forward_packed_batched(W, ids[:, i:i + step].contiguous(), st2).view(
            B, -1, whole.shape[-1]) for i in range(0, T, step)]
        assert torch.equal(whole, torch.cat(parts, 1))
        assert torch.equal(st.buf, st2.buf)
    finally:
        cpp_path.release_weights(w)
