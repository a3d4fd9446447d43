"""Nodal proposals of nodes whose lists end at the edges of k_nodal's paths: the
1, 2 and 4 entries a lane holds (64, 128, 256), nodes the whole workgroup takes
with its table in LDS and beyond (1536 units), on M all direct and hashed,
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 384, 385, 1200, 1537, 3001]


def _graph(usap, weighted, N=2400):
    """Node i has SIZES[i] list entries (out and in mixed, a few self-loops);
    the other nodes are sparse."""
    rng = np.random.default_rng(17)
    src, dst = [rng.integers(len(SIZES), N, 4000)], [rng.integers(len(SIZES), N, 4000)]
    for i, k in enumerate(SIZES):
        loops = 1 if k >= 64 else 0  # a self-loop is two list entries
        out = (k - 2 * loops) // 2
        other = rng.integers(len(SIZES), N, k - 2 * loops)
        src += [np.full(out + loops, i), other[out:]]
        dst += [np.concatenate([other[:out], np.full(loops, i)]), np.full(k - 2 * loops - out, i)]
    src, dst = np.concatenate(src), np.concatenate(dst)
    perm = rng.permutation(len(src))
    src, dst = src[perm], dst[perm]
    w = rng.integers(0, 4, len(src)) if weighted else None
    g = usap.Graph.from_edges(src, dst, N, w)
    got = np.diff(g.out_ptr)[:len(SIZES)] + np.diff(g.in_ptr)[:len(SIZES)]
    np.testing.assert_array_equal(got, SIZES)
    return g


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("B", [3, 40, 1500, 2400])
def test_list_sizes(usap, orc, weighted, mode, B):
    g = _graph(usap, weighted)
    lab = np.random.default_rng(B).permutation(np.arange(g.N) % B).astype(np.int32)
    eng = usap.Engine(g, seed=5, ds_mode=mode)
    o = orc.Oracle(g, threads=8, seed=5, ds_mode=mode)
    eng.set_labels(lab, B)
    o.set_labels(lab, B)
    n = len(SIZES) + 8
    for stream in range(6):  # many draws of every node: both proposal branches
        r, ro = eng.nodal_batch(0, n, stream), o.nodal_batch(0, n, stream)
        np.testing.assert_array_equal(r["s"], ro["s"])
        np.testing.assert_array_equal(r["accept"], ro["accept"])
        np.testing.assert_array_equal(r["inf"], np.where(ro["inf"] == -1, -1, 0))
        fin = ro["inf"] == 0
        assert [x for x, f in zip(r["dS"], fin) if f] == [x for x, f in zip(ro["dS"], fin) if f]
        assert r["sum"] == ro["sum"]
        np.testing.assert_array_equal(eng.labels(), o.labels())
    assert eng.entropy()[0] == o.entropy()[0]
    np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
