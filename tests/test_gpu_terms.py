"""The dS and MDL term sums (two split products per term) against the oracle's
int128 ones, exactly, at weights where both parts of the split carry many bits
and the row sums approach the total weight."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("B", [2, 37, 150])
def test_large_weights(usap, orc, mode, B):
    rng = np.random.default_rng(B)
    N = 150
    src, dst = rng.integers(0, N, 1500), rng.integers(0, N, 1500)
    w = rng.integers(0, 2, 1500) * rng.integers(1, 40000, 1500)  # weight 0 among them
    w[:3] = 1 << 22
    g = usap.Graph.from_edges(src, dst, N, w)
    lab = (np.arange(N) % B).astype(np.int32)
    eng = usap.Engine(g, seed=3, ds_mode=mode)
    o = orc.Oracle(g, threads=4, seed=3, ds_mode=mode)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    assert eng.entropy()[0] == o.entropy()[0]
    s, d = eng.merge_propose(0)
    os_, od = o.block_merge(0)
    np.testing.assert_array_equal(s, os_)
    assert d == od
    for i, beg in enumerate(range(0, N, 50)):
        r, ro = eng.nodal_batch(beg, beg + 50, i), o.nodal_batch(beg, beg + 50, i)
        np.testing.assert_array_equal(r["s"], ro["s"])
        np.testing.assert_array_equal(r["accept"], ro["accept"])
        fin = ro["inf"] == 0
        assert [x for x, f in zip(r["dS"], fin) if f] == [x for x, f in zip(ro["dS"], fin) if f]
        assert r["sum"] == ro["sum"]
    assert eng.entropy()[0] == o.entropy()[0]
