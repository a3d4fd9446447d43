"""The M build at B = N (a search's start from one block per node) where the block
counts below it are built another way: one node per block, and as many blocks
with some of them empty; M, degrees, the MDL, a nodal batch and a merge round
against the oracle."""
import numpy as np
import pytest

from conftest import random_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("N,E", [(257, 900), (300, 20000), (513, 4000), (1100, 9000), (4096, 30000)])
def test_as_many_blocks_as_nodes(usap, orc, N, E, weighted):
    g = random_graph(N, E, seed=N, weighted=weighted, self_loops=True, hubs=1, isolated=7)
    rng = np.random.default_rng(N)
    eng = usap.Engine(g, seed=2, K=3)
    o = orc.Oracle(g, threads=8, seed=2, K=3)
    for lab in (np.arange(N), rng.permutation(N), rng.integers(0, N, N)):
        lab = lab.astype(np.int32)
        eng.set_labels(lab, N)
        o.set_labels(lab, N)
        np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
        for a, b in zip(eng.degrees(), o.degrees()):
            np.testing.assert_array_equal(a, b)
        assert eng.entropy()[0] == o.entropy()[0]
        s, d = eng.merge_propose(1)
        so, do = o.block_merge(1)
        np.testing.assert_array_equal(s, so)
        assert d == do
        r, ro = eng.nodal_batch(0, N, 1), o.nodal_batch(0, N, 1)
        np.testing.assert_array_equal(r["s"], ro["s"])
        np.testing.assert_array_equal(eng.labels(), o.labels())
        np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
