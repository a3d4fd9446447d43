"""Rows of M growing between batches across the sizes k_grow and the pick treat
apart: slabs a wavefront handles (up to 512 slots, new slab up to 1024), those
of the workgroup, hashed rows that become direct, rows that start to keep
bucket sums; against the oracle, batch by batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slack", [1, 2])
def test_growth_across_row_sizes(usap, orc, slack):
    rng = np.random.default_rng(23)
    N, B = 19000, 17000
    # blocks of 1 node, and sixty of 2 to 60 nodes whose members have more edges
    sizes = np.ones(B, int)
    sizes[:60] += np.linspace(1, 66, 60).astype(int)
    sizes[0] += N - sizes.sum()
    lab = np.repeat(np.arange(B), sizes).astype(np.int32)
    heavy = np.flatnonzero(lab < 60)
    src = np.concatenate([rng.integers(0, N, 30000), rng.choice(heavy, 25000)])
    dst = np.concatenate([rng.integers(0, N, 30000), rng.integers(0, N, 25000)])
    g = usap.Graph.from_edges(src, dst, N)
    eng = usap.Engine(g, seed=9, slab_slack=slack)
    o = orc.Oracle(g, threads=16, seed=9)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    for i, beg in enumerate(range(0, 12000, 1500)):
        r, ro = eng.nodal_batch(beg, beg + 1500, i), o.nodal_batch(beg, beg + 1500, i)
        np.testing.assert_array_equal(r["s"], ro["s"])
        np.testing.assert_array_equal(r["accept"], ro["accept"])
        fin = ro["inf"] == 0
        assert [x for x, f in zip(r["dS"], fin) if f] == [x for x, f in zip(ro["dS"], fin) if f]
        assert eng.entropy()[0] == o.entropy()[0]
    np.testing.assert_array_equal(eng.labels(), o.labels())
    # a merge round reads every row, the grown ones' bucket sums among them
    s, d = eng.merge_propose(3)
    os_, od = o.block_merge(3)
    np.testing.assert_array_equal(s, os_)
    assert d == od
