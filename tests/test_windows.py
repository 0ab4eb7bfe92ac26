"""Packed windows over streams of different lengths: the plan covers every
stream, and a payload does not depend on the streams compressed beside it."""
import numpy as np
import pytest

from krunch_amd import synthetic
from krunch_amd.inference import InferenceEngine, plan_windows

LENS = [[1], [1, 1], [1024] * 3, [1025, 1024, 1], [1300, 999, 700, 325], [5000, 64, 64, 63, 1],
        list(range(300, 0, -1)), [3000] * 200 + [1], [17, 16, 1]]


@pytest.mark.parametrize("window", [1, 7, 100, 1024])
@pytest.mark.parametrize("lens", LENS, ids=lambda v: f"{len(v)}x{v[0]}")
def test_plan_covers_every_stream(lens, window):
    lens = np.array(lens)
    plan = plan_windows(lens, window)
    assert plan[0][0] == 0 and plan[-1][1] == lens[0] and plan[0][2] == len(lens)
    for (a, b, n), nxt in zip(plan, plan[1:] + [(lens[0], 0, 0)]):
        assert b == nxt[0] and 1 <= b - a <= window
        assert n == int((lens > a).sum())
    if lens[-1] == lens[0]:
        assert [p[0] for p in plan] == list(range(0, int(lens[0]), window))


# streams that end at a cut, one past it and one before it, order reversed and
# mixed, more streams than one short stream each; both codecs
@pytest.mark.gpu
@pytest.mark.parametrize("w8a8", [False, True])
@pytest.mark.parametrize("window,lens", [(1024, [3, 700, 64, 65, 63, 700, 1]), (96, [40, 97, 300, 6, 12, 299, 13]),
                                         (1024, [1500, 1024, 1025, 128] + [200] * 24)])
def test_payloads_do_not_depend_on_the_batch(lens, window, w8a8):
    e = InferenceEngine().load(synthetic.make_weights(n_layer=2, V=1000), w8a8=w8a8)
    e.window = window
    toks = [synthetic.zipf_tokens(1, n, V=1000, seed_base=i)[0] for i, n in enumerate(lens)]
    got = e.compress_tokens_batched(toks)
    assert got == [e.compress_tokens_batched([t])[0] for t in toks]
    for t, d in zip(toks, e.decompress_tokens_batched(got)):
        np.testing.assert_array_equal(t, d)
