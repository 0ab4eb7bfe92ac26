"""The head's C entry: LN_out scratch in place of its input, and the row counts
and strides where its kernels meet."""
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


# both sides of each line between the register-held rows and the 256 x 256
# tiles: strides of whole 4096 bytes, few columns, output size at the small
# widths, row groups that fill the CUs, several launches
@pytest.mark.parametrize("C,V,ld,Ms", [(256, 2040, 2048, (1024, 1040)), (768, 1000, 1000, (4096, 4112)),
                                       (512, 5000, 5000, (8192, 8208)), (256, 40000, 40000, (2496, 2512)),
                                       (768, 5000, 5000, (5120, 6144)), (768, 20000, 20000, (8208,)),
                                       (256, 4097, 4097, (8208,)), (256, 1001, 1001, (8192, 8208))])
def test_head_on_both_sides_of_its_lines(C, V, ld, Ms):
    """The head's kernels share one contract: a row's logits do not depend on
    the rows around it (here against 512 rows at a time)."""
    w = synthetic.make_weights(n_layer=1, C=C, F=256, V=V, seed=C + V)
    P = cpp_path.init_weights(w, "cuda")["prepared"]
    try:
        for M in Ms:
            x = torch.randn((M, C), generator=torch.Generator().manual_seed(M)).half().cuda()
            got = _head(P, x, torch.empty_like(x), ld)
            for r in range(0, M, 512):
                part = x[r:r + 512].contiguous()
                assert torch.equal(got[r:r + 512], _head(P, part, torch.empty_like(part), ld)), (M, r)
    finally:
        cpp_path.release_weights(w)


# one row, around a 16-row block, around the decode head's 512 rows; widths
# with and without fragment-packed heads
@pytest.mark.parametrize("C", [256, 1024])
@pytest.mark.parametrize("M", [1, 15, 17, 511, 513, 700])
def test_logits_hold_their_rows_only(C, M):
    """Packed and stepped logits own M rows and no more, equal to the head's
    over rows of their own."""
    w = synthetic.make_weights(n_layer=1, C=C, F=256, V=1003, seed=M)
    W = cpp_path.init_weights(w, "cuda")
    try:
        ids = torch.from_numpy(synthetic.zipf_tokens(1, M, V=1003))
        got = cpp_path.forward_packed_batched(W, ids, cpp_path.fresh_state(W))
        assert got.shape == (M, 1003) and got.untyped_storage().nbytes() == 2 * M * 1003
        st = cpp_path.fresh_state(W)
        for t in range(min(M, 3)):
            one = cpp_path.forward_stepped(W, int(ids[0, t]), st)
            assert torch.equal(one, got[t]) and one.untyped_storage().nbytes() == 2 * 1003
        st.reset()
        assert torch.equal(cpp_path.forward_stepped_graphed(W, int(ids[0, 0]), st), got[0])
    finally:
        cpp_path.clear_graph_cache()
        cpp_path.release_weights(w)
