"""Merge proposals of blocks whose rows end at the edges of the two kernels: 64,
255 to 257 and 511 to 513 non-zero keys, slabs of 1024 slots and above, direct rows among
hashed ones, a workgroup's 4 and 16 wavefronts, and more proposals than a
wavefront has lanes, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = [0, 1, 63, 64, 65, 255, 256, 257, 300, 500, 503, 511, 512, 513, 600, 1100, 3000]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("K", [1, 10, 70])
@pytest.mark.parametrize("B", [3, 900, 1100, 18000])
def test_merge_rows(usap, orc, B, K, weighted):
    rng = np.random.default_rng(B + K)
    N = B + 50
    lab = np.concatenate([np.arange(B), rng.integers(0, B, N - B)]).astype(np.int32)
    src, dst = [rng.integers(len(KEYS), N, 2 * N)], [rng.integers(len(KEYS), N, 2 * N)]
    for i, k in enumerate(KEYS):
        if i >= B or k > B - 20:
            continue
        # the first of them are keys of several of these rows: overlaps that count
        other = np.concatenate([np.arange(20, 20 + min(k, 40)) % B,
                                rng.choice(np.arange(60, B), max(k - 40, 0), replace=False)
                                if k > 40 else np.zeros(0, np.int64)])
        half = k // 2
        src += [np.full(half, i), other[half:]]
        dst += [other[:half], np.full(k - half, i)]
    src, dst = np.concatenate(src), np.concatenate(dst)
    perm = rng.permutation(len(src))
    src, dst = src[perm], dst[perm]
    w = rng.integers(1, 400, len(src)) if weighted else None
    g = usap.Graph.from_edges(src, dst, N, w)
    eng = usap.Engine(g, seed=3, K=K)
    o = orc.Oracle(g, threads=8, seed=3, K=K)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    for stream in range(3):
        s, d = eng.merge_propose(stream)
        so, do = o.block_merge(stream)
        np.testing.assert_array_equal(s, so)
        assert d == do
