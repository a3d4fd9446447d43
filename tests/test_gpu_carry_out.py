"""The carry-out on the device (one workgroup with ranks by comparison, one
workgroup after a sort, the whole GPU) against the reference's loop restated
over a round's own proposals: labels for every number of merges up to running
out of candidates."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _greedy(s, dS, n):
    """graph_parallel.hpp:1225-1279: (map of the blocks, links possible)."""
    B = len(s)
    parent = np.arange(B)

    def find(x):
        while parent[x] != x:
            parent[x] = parent[parent[x]]
            x = parent[x]
        return x

    made = 0
    for i in sorted(range(B), key=lambda b: (dS[b], b)):
        if made == n:
            break
        to = find(s[i])
        if to != i:
            parent[i] = to
            made += 1
    roots = np.array([find(b) for b in range(B)])
    return np.unique(roots, return_inverse=True)[1], made


@pytest.mark.parametrize("B", [2, 3, 64, 1000, 1024, 1025, 5000, 8192, 8193, 20000])
def test_carry_out(usap, B):
    rng = np.random.default_rng(B)
    N = B + B // 8
    src, dst = rng.integers(0, N, 3 * N), rng.integers(0, N, 3 * N)
    # a path and a star, whose proposals chain and share one target
    src = np.concatenate([src, np.arange(N // 4), np.full(N // 8, N - 1)])
    dst = np.concatenate([dst, np.arange(1, N // 4 + 1), rng.integers(0, N, N // 8)])
    g = usap.Graph.from_edges(src, dst, N)
    lab = np.concatenate([np.arange(B), rng.integers(0, B, N - B)]).astype(np.int32)
    eng = usap.Engine(g, seed=B)
    most = None
    for n in (0, 1, B // 3, B // 2, (9 * B) // 10, B - 1):
        if n >= B:
            continue
        eng.set_labels(lab, B)
        s, dS = eng.merge_propose(1, K=3)
        want, made = _greedy(s, dS, n)
        if made < n:  # out of candidates: refused, nothing changed
            with pytest.raises(Exception, match="candidate"):
                eng.merge_apply(n)
            np.testing.assert_array_equal(eng.labels(), lab)
            assert eng.B == B
            n = made
            assert eng.merge_apply(n) == B - n
            want, _ = _greedy(s, dS, n)
        else:
            assert eng.merge_apply(n) == B - n
        np.testing.assert_array_equal(eng.labels(), want[lab])
        do, di = eng.degrees()
        np.testing.assert_array_equal(do, np.bincount(want[lab][src], minlength=B - n))
        np.testing.assert_array_equal(di, np.bincount(want[lab][dst], minlength=B - n))
