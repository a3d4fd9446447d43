"""The M build for few blocks (histograms in LDS, one or two halves of the rows)
and the build just above it, at the sizes where the path changes: M, degrees,
sizes through the next merge, and the MDL against counts of the labels."""
import numpy as np
import pytest

from conftest import random_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("B", [1, 2, 63, 64, 65, 128, 129, 200, 201, 255, 256, 257])
def test_build(usap, orc, B, weighted):
    E = 30000 if B % 2 else 300  # several workgroups' shares, or one
    g = random_graph(700, E, seed=B, weighted=weighted, self_loops=True, hubs=1, isolated=9)
    lab = (np.random.default_rng(B).permutation(g.N) % B).astype(np.int32)
    eng = usap.Engine(g, seed=2)
    o = orc.Oracle(g, threads=4, seed=2)
    for _ in range(2):  # the second build finds the first one's state
        eng.set_labels(lab, B)
        o.set_labels(lab, B)
        np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
        for a, b in zip(eng.degrees(), o.degrees()):
            np.testing.assert_array_equal(a, b)
        assert eng.entropy()[0] == o.entropy()[0]
        r, ro = eng.nodal_batch(0, g.N, 1), o.nodal_batch(0, g.N, 1)
        np.testing.assert_array_equal(r["s"], ro["s"])
        np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
        if B > 1:
            s, d = eng.merge_propose(0)
            os_, od = o.block_merge(0)
            np.testing.assert_array_equal(s, os_)
            assert d == od
            eng.merge_apply(B // 2)
            assert o.carry_out(B // 2) == 0
            np.testing.assert_array_equal(eng.labels(), o.labels())
            np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
        lab = lab[::-1].copy()


def test_no_edges(usap):
    g = usap.Graph.from_edges(np.zeros(0, np.int32), np.zeros(0, np.int32), 12)
    eng = usap.Engine(g, seed=2)
    eng.set_labels((np.arange(12) % 3).astype(np.int32), 3)
    assert not eng.M_dense().any()
    assert not eng.degrees()[0].any() and not eng.degrees()[1].any()
