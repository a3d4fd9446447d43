"""Edge arrays of other types than int32 reach the library whole: the converted
copies live until the call has read them."""
import ctypes as C

import numpy as np
import pytest

from usap_amd import engine


class _Lib:
    """usap_create_from_edges and usap_append_edges that read what they are given."""

    def __init__(self):
        self.seen = []

    def _read(self, n, *ptrs):
        np.empty(4 * n, np.int8).fill(77)  # what a freed copy may be used for
        self.seen.append([None if p is None else
                          np.ctypeslib.as_array((C.c_int32 * n).from_address(p)).tolist()
                          for p in ptrs])

    def usap_default_params(self, p):
        pass

    def usap_create_from_edges(self, N, E, src, dst, w, params, out):
        self._read(E, src, dst, w)
        return 0

    def usap_append_edges(self, h, n, src, dst, w):
        self._read(n, src, dst, w)
        return 0

    def usap_destroy(self, h):
        return 0


@pytest.mark.parametrize("dtype", [np.int64, np.int32, np.uint8, list])
def test_edges_of_any_type(monkeypatch, dtype):
    lib = _Lib()
    monkeypatch.setattr(engine, "lib", lambda: lib)
    src, dst, w = [np.arange(k, k + 50) for k in (0, 50, 100)]
    want = [x.tolist() for x in (src, dst, w)]
    edges = tuple(x.tolist() if dtype is list else x.astype(dtype) for x in (src, dst, w))

    class G:
        N = 200

    e = engine.Engine(G, edges=edges)
    e.append_edges(*edges)
    e.append_edges(*edges[:2])
    assert lib.seen == [want, want, want[:2] + [None]]
    e.h = None
