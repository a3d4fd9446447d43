"""The M build by rows with nodes whose lists are split over workgroups: at the
edges of a part (8192 list entries), many parts, several such nodes in one block,
one that reaches the size by appended edges; against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ENTRIES = [8191, 8192, 8193, 16384, 16385, 100001]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("B", [300, 4200, 6000])
def test_huge_lists(usap, orc, B, weighted):
    rng = np.random.default_rng(B + weighted)
    N = 300 if B == 300 else 6000
    n = len(ENTRIES)
    src, dst = [rng.integers(n, N, 8000)], [rng.integers(n, N, 8000)]
    for i, k in enumerate(ENTRIES):
        out = k // 3
        src += [np.full(out, i), rng.integers(n, N, k - out)]
        dst += [rng.integers(n, N, out), np.full(k - out, i)]
    late = 9000  # the edges appended at the end: node n's
    src.append(np.full(late, n))
    dst.append(rng.integers(n + 1, N, late))
    src, dst = np.concatenate(src), np.concatenate(dst)
    perm = rng.permutation(len(src) - late)
    src[:-late], dst[:-late] = src[perm], dst[perm]
    w = rng.integers(0, 4, len(src)).astype(np.int32) if weighted else None
    g = usap.Graph.from_edges(src, dst, N, w)
    entries = np.diff(g.out_ptr) + np.diff(g.in_ptr)
    np.testing.assert_array_equal(entries[:n], ENTRIES)
    eng = usap.Engine(g, seed=2, edges=(src[:-late], dst[:-late], None if w is None else w[:-late]))
    o = orc.Oracle(g, threads=8, seed=2)
    lab = (rng.permutation(N) % B).astype(np.int32)
    lab[:3] = lab[3]  # several in one block
    eng.set_labels(lab, B)
    eng.append_edges(src[-late:], dst[-late:], None if w is None else w[-late:])
    o.set_labels(lab, B)
    for labels in (lab, rng.permutation(B).astype(np.int32)[lab]):
        eng.set_labels(labels, B)
        o.set_labels(labels, B)
        for x, y in zip(eng.degrees(), o.degrees()):
            np.testing.assert_array_equal(x, y)
        assert eng.entropy()[0] == o.entropy()[0]
        np.testing.assert_array_equal(eng.M_dense(), o.M_dense())
    r, ro = eng.nodal_batch(0, 40, 1), o.nodal_batch(0, 40, 1)
    np.testing.assert_array_equal(r["s"], ro["s"])
    np.testing.assert_array_equal(eng.labels(), o.labels())
