"""Captured sweeps (graphs=1) of one block count whose M changes between all
rows direct and some hashed: at B > 256 that follows the labels (a block of few
edges has a hashed row), and setting labels again at the same B need not
allocate.  Moves, dS, labels and M of every sweep against the oracle."""
import numpy as np
import pytest

from conftest import random_graph

pytestmark = pytest.mark.gpu


def _entries(g, lab, B):
    deg = np.diff(g.out_ptr) + np.diff(g.in_ptr)
    return np.bincount(lab, weights=deg, minlength=B)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("order", ["direct first", "hashed first"])
@pytest.mark.parametrize("B,most_hashed", [(300, 8), (600, 24)])
def test_replay_follows_the_rows(usap, orc, B, most_hashed, order, weighted):
    g = random_graph(1500, 30000, seed=B, weighted=weighted, self_loops=True, isolated=12)
    rng = np.random.default_rng(B)
    direct = rng.permutation(np.arange(g.N) % B).astype(np.int32)
    while _entries(g, direct, B).min() <= most_hashed:  # isolated nodes may share a block
        direct = rng.permutation(direct)
    # the isolated nodes in block 0, whose hashed row comes first
    hashed = (1 + np.arange(g.N) % (B - 1)).astype(np.int32)
    hashed[-12:] = 0
    assert _entries(g, hashed, B)[0] == 0 and _entries(g, hashed, B)[1:].min() > most_hashed
    eng = usap.Engine(g, seed=6, graphs=1)
    o = orc.Oracle(g, threads=4, seed=6)
    # the largest M first, so that no later build has to allocate
    eng.set_labels(direct, B)
    first, second = (direct, hashed) if order == "direct first" else (hashed, direct)
    batch, stream = 400, 0
    for lab in (first, second, first, second, second):
        eng.set_labels(lab, B)
        o.set_labels(lab, B)
        a = eng.nodal_sweep(batch, stream, 0.0, 0.0, 0.0, 0)
        moves = total = 0
        inf = False
        for i, beg in enumerate(range(0, g.N, batch)):
            r = o.nodal_batch(beg, min(beg + batch, g.N), stream + i)
            moves += r["moves"]
            inf = inf or bool(r["sum_inf"])
            total += 0 if r["sum_inf"] else r["sum"]
        assert a["moves"] == moves
        assert inf or a["dS_fx"] == total
        np.testing.assert_array_equal(eng.labels(), o.labels())
        np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
        for x, y in zip(eng.degrees(), o.degrees()):
            np.testing.assert_array_equal(x, y)
        assert eng.entropy()[0] == o.entropy()[0]
        stream += a["batches"]
