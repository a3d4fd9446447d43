"""Merge proposals where k_merge_rows leaves most blocks to k_merge: more of them
than k_merge has workgroups, long rows (direct, beyond what is looked through)
and shorter ones in several workgroups of the list, with proposals as many as a
workgroup's wavefronts and one more, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("K", [1, 4, 5])
def test_many_rows_left(usap, orc, K, weighted):
    rng = np.random.default_rng(K)
    B, N = 9000, 9100
    lab = np.concatenate([np.arange(B), rng.integers(0, B, N - B)]).astype(np.int32)
    # 160 edges out of every node but 200 (their rows stay short), and the first 40
    # blocks' rows long
    few = rng.choice(np.arange(40, B), 200, replace=False)
    many = np.setdiff1d(np.arange(N), few)
    src, dst = np.repeat(many, 160), rng.choice(many, 160 * len(many))
    src = np.concatenate([src, few, np.repeat(np.arange(40), 500)])
    dst = np.concatenate([dst, rng.integers(0, N, len(few)), rng.integers(0, N, 40 * 500)])
    w = rng.integers(1, 5, len(src)) if weighted else None
    g = usap.Graph.from_edges(src, dst, N, w)
    entries = np.bincount(lab, weights=np.diff(g.out_ptr) + np.diff(g.in_ptr), minlength=B)
    # slabs of 1024 slots up to 504 list entries, direct rows of 9000 beyond
    assert (entries > 504).sum() >= 40
    assert ((entries > 270) & (entries <= 504)).sum() + (entries > 504).sum() > 8192 + 512
    eng = usap.Engine(g, seed=3, K=K)
    o = orc.Oracle(g, threads=8, seed=3, K=K)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    for stream in range(2):
        s, d = eng.merge_propose(stream)
        so, do = o.block_merge(stream)
        np.testing.assert_array_equal(s, so)
        assert d == do
