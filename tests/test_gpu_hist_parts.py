"""The M build for few blocks at edge counts that give k_hist_sum more parts than
one group of threads, more than one round of all groups, with a remainder, and
the most there are (256, or 128 a half): M and degrees against counts of the
labels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("E", [4096 * 9 + 5, 4096 * 33 + 1, 4096 * 129, 4096 * 257 + 3])
@pytest.mark.parametrize("B", [1, 33, 129, 200, 201, 256])
def test_parts(usap, B, E, weighted):
    rng = np.random.default_rng(B)
    N = 3000
    src, dst = rng.integers(0, N, E), rng.integers(0, N, E)
    w = rng.integers(0, 5, E).astype(np.int32) if weighted else None
    eng = usap.Engine(usap.Graph.from_edges(src, dst, N, w), seed=2)
    lab = rng.integers(0, B, N).astype(np.int32)
    eng.set_labels(lab, B)
    want = np.bincount(lab[src].astype(np.int64) * B + lab[dst], weights=w,
                       minlength=B * B).reshape(B, B).astype(np.int64)
    np.testing.assert_array_equal(eng.M_dense(), want)
    do, di = eng.degrees()
    np.testing.assert_array_equal(do, want.sum(1))
    np.testing.assert_array_equal(di, want.sum(0))
