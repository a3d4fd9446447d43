"""Sweeps whose marked rows wait for k_grow's next look, over one look, up to the
next and past it (8 batches apart), against the oracle's batches."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slack", [1, 2])
@pytest.mark.parametrize("batches", [1, 8, 9, 10, 25])
def test_sweep(usap, orc, slack, batches):
    rng = np.random.default_rng(batches)
    N, B = 9000, 6000
    lab = np.concatenate([np.arange(B), rng.integers(0, 40, N - B)]).astype(np.int32)
    heavy = np.flatnonzero(lab < 40)
    src = np.concatenate([rng.integers(0, N, 20000), rng.choice(heavy, 15000)])
    dst = np.concatenate([rng.integers(0, N, 20000), rng.integers(0, N, 15000)])
    g = usap.Graph.from_edges(src, dst, N)
    eng = usap.Engine(g, seed=4, slab_slack=slack)
    o = orc.Oracle(g, threads=8, seed=4)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    size = -(-N // batches)
    eng.nodal_sweep(size, 0, 1e6, 0.0, 1e-4, False)
    for i, beg in enumerate(range(0, N, size)):
        o.nodal_batch(beg, min(beg + size, N), i)
    np.testing.assert_array_equal(eng.labels(), o.labels())
    assert eng.entropy()[0] == o.entropy()[0]
    s, d = eng.merge_propose(3)
    so, do = o.block_merge(3)
    np.testing.assert_array_equal(s, so)
    assert d == do
