"""Packed windows of a few hundred to a few thousand rows (fragment-packed
operands through the register-fed product kernel) against the same tokens in
windows of at most 512 rows, which the small-M kernels run: the reduction
contract makes them equal bit for bit, state included."""
import pytest
import torch

from krunch_amd import cpp_path, krunch_ac_hip, synthetic

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
