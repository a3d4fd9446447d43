"""Graphs whose edges weigh nothing (none at all, or all of weight 0), for which
lambda's table is its entry 0 alone: nodal batches, a sweep, merge rounds and the
data term on M all direct and hashed, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("edges", [0, 3000])
@pytest.mark.parametrize("B", [1, 3, 400, 5000])
def test_no_weight(usap, orc, B, edges, mode):
    rng = np.random.default_rng(B)
    N = max(B, 500)
    src, dst = rng.integers(0, N, edges), rng.integers(0, N, edges)
    src[:edges // 2] = 7  # one node the whole workgroup takes
    g = usap.Graph.from_edges(src, dst, N, np.zeros(edges, np.int32) if edges else None)
    lab = (rng.permutation(N) % B).astype(np.int32)
    eng = usap.Engine(g, seed=4, ds_mode=mode, K=3)
    o = orc.Oracle(g, threads=4, seed=4, ds_mode=mode, K=3)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    for stream in range(3):
        r, ro = eng.nodal_batch(0, N, stream), o.nodal_batch(0, N, stream)
        np.testing.assert_array_equal(r["s"], ro["s"])
        np.testing.assert_array_equal(r["accept"], ro["accept"])
        assert r["dS"] == ro["dS"] and r["sum"] == ro["sum"] == 0
        if B > 1:
            s, d = eng.merge_propose(stream)
            so, do = o.block_merge(stream)
            np.testing.assert_array_equal(s, so)
            assert d == do
    sw = eng.nodal_sweep(max(1, N // 4), 9, 0.0, 0.0, 0.0, 0)
    assert sw["dS_fx"] == 0
    np.testing.assert_array_equal(eng.degrees()[0], np.zeros(B, np.int32))
    assert eng.M_coo()[0].size == 0
    assert eng.entropy()[0] == 0
