"""The M build by rows (B above 4096): slabs of up to 256 and up to 1024 slots,
direct rows, a block of thousands of nodes, a hub whose list is split over
workgroups, a block with more neighbour blocks than its LDS table, one block per
node, empty blocks' rows; against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("B,N", [(4096, 9000), (4097, 9000), (4500, 70000), (17000, 26000),
                                 (9000, 9000)])
def test_row_build(usap, orc, B, N, weighted):
    rng = np.random.default_rng(B + weighted)
    src, dst = [rng.integers(0, N, 4 * N)], [rng.integers(0, N, 4 * N)]
    for hub, k in ((5, 20000), (6, 3000), (7, 500)):
        src.append(np.full(k, hub))
        dst.append(rng.integers(0, N, k))
    for k in range(40):  # lists on both sides of 256 and 1024 slots
        src.append(rng.integers(0, N, 8 * k))
        dst.append(np.full(8 * k, 100 + k))
    src, dst = np.concatenate(src), np.concatenate(dst)
    perm = rng.permutation(len(src))
    src, dst = src[perm], dst[perm]
    w = rng.integers(0, 50, len(src)) if weighted else None
    g = usap.Graph.from_edges(src, dst, N, w)
    # block 3 has most of the nodes beyond the first B
    more = np.where(rng.random(N - B) < 0.7, 3, rng.integers(0, B, N - B))
    lab = np.concatenate([np.arange(B), more]).astype(np.int32)
    eng = usap.Engine(g, seed=2)
    o = orc.Oracle(g, threads=8, seed=2)
    for labels in (lab, rng.permutation(B).astype(np.int32)[lab]):
        eng.set_labels(labels, B)
        o.set_labels(labels, B)
        for x, y in zip(eng.degrees(), o.degrees()):
            np.testing.assert_array_equal(x, y)
        assert eng.entropy()[0] == o.entropy()[0]
        if B < 4500:
            np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
        s, d = eng.merge_propose(1)
        so, do = o.block_merge(1)
        np.testing.assert_array_equal(s, so)
        assert d == do


def test_no_edges(usap):
    N = 5000
    g = usap.Graph.from_edges(np.zeros(0, np.int32), np.zeros(0, np.int32), N)
    eng = usap.Engine(g, seed=2)
    eng.set_labels(np.arange(N, dtype=np.int32), N)
    assert all(not x.any() for x in eng.degrees())
    assert eng.M_dense().sum() == 0
