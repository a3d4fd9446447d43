"""usap_footprint against what engines take from the device's memory pool: a
partition from one block per node, one from the default start with edges
appended, a graph with one very large node, a dense one."""
import ctypes as C

import numpy as np
import pytest

from usap_amd import serve as sv

pytestmark = pytest.mark.gpu

USED, USED_HIGH = 7, 8  # hipMemPoolAttrUsedMemCurrent, hipMemPoolAttrUsedMemHigh


class _Pool:
    """The device's default pool, by the runtime that the library is linked to."""

    def __init__(self):
        path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
        self.hip, self.h = C.CDLL(path), C.c_void_p()
        assert self.hip.hipDeviceGetDefaultMemPool(C.byref(self.h), 0) == 0

    def get(self, attr):
        v = C.c_uint64()
        assert self.hip.hipMemPoolGetAttribute(self.h, attr, C.byref(v)) == 0
        return v.value

    def reset_high(self):
        assert self.hip.hipMemPoolSetAttribute(self.h, USED_HIGH, C.byref(C.c_uint64(0))) == 0


def _graph(usap, kind):
    rng = np.random.default_rng(3)
    if kind == "star":
        N = 20000
        src = np.concatenate([rng.integers(0, N, 40000), np.zeros(100000, np.int64)])
        return usap.Graph.from_edges(src, rng.integers(0, N, len(src)), N)
    if kind == "dense":
        return usap.Graph.from_edges(rng.integers(0, 2000, 300000), rng.integers(0, 2000, 300000), 2000)
    N = int(kind)
    return usap.generate_dcsbm(N, 10, 3.0, 20, 10, min(100, N // 4), 2.5, 0.7, 1)


@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("kind", ["500", "5000", "50000", "star", "dense"])
def test_footprint_holds(usap, kind, append):
    g = _graph(usap, kind)
    usap.Engine(g).close()  # the library and its pool are there
    pool = _Pool()
    before = pool.get(USED)
    pool.reset_high()
    if append:
        src, dst = (x.astype(np.int32) for x in g.edges())
        k = len(src) // 2
        eng = usap.Engine(g, edges=(src[:k], dst[:k], None), seed=1)
        eng.partition()
        eng.append_edges(src[k:], dst[k:])
    else:
        eng = usap.Engine(g, seed=1, init=1)
    eng.partition()
    used = pool.get(USED_HIGH) - before
    eng.close()
    assert 0 < used <= sv.footprint(g.N, g.E)
