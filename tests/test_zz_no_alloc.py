"""The allocation-free neighbour search (sph_ns_find_neighbors_noalloc)
against the drop-in search (sph_ns_find_neighbors + sph_ns_neighbor_csr) on
the same points: identical CSR arrays, on two calls in a row (the second
with fewer points, so stale scratch contents from the first would show), a
too-small output buffer, an empty set and a size beyond the maximum."""
import ctypes as C

import numpy as np
import pytest

from splishsplash_amd import capi

pytestmark = pytest.mark.gpu

SPH_ERR_RANGE = -7


def cloud(n, seed):
    rng = np.random.default_rng(seed)
    # half uniform, half in a few tight clusters: cells of very different sizes
    u = rng.random((n - n // 2, 3))
    c = rng.random((8, 3)) * 0.8 + 0.1
    k = rng.integers(0, 8, n // 2)
    g = c[k] + rng.normal(scale=0.02, size=(n // 2, 3))
    return np.ascontiguousarray(np.vstack([u, g]).astype(np.float32))


def drop_in(x, radius):
    ns = capi.NeighborhoodSearch(radius)
    ns.add_point_set(x)
    ns.find_neighbors()
    off, idx = ns.neighbors_csr(0, 0)
    del ns
    return off, idx


class Hip:
    """The HIP runtime the library itself runs on (its libamdhip64.so.7,
    already loaded with it), for the device buffers of the test."""

    def __init__(self):
        capi.lib()
        self.L = C.CDLL("libamdhip64.so.7")
        self.L.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.L.hipFree.argtypes = [C.c_void_p]
        self.L.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]

    def alloc(self, nbytes):
        p = C.c_void_p()
        assert self.L.hipMalloc(C.byref(p), max(int(nbytes), 4)) == 0
        return p

    def put(self, dst, a):
        assert self.L.hipMemcpy(dst, a.ctypes.data, a.nbytes, 1) == 0  # host to device

    def get(self, src, a):
        assert self.L.hipMemcpy(a.ctypes.data, src, a.nbytes, 2) == 0  # device to host
        return a

    def free(self, *ps):
        for p in ps:
            self.L.hipFree(p)


def noalloc(x, radius, capacity):
    hip = Hip()
    n = len(x)
    xd, od, nd = hip.alloc(12 * n), hip.alloc(4 * (n + 1)), hip.alloc(4 * max(capacity, 1))
    try:
        hip.put(xd, np.ascontiguousarray(x, np.float32).reshape(-1))
        hip.put(od, np.full(n + 1, 0xFFFFFFFF, np.uint32))
        total = C.c_size_t(0)
        rc = capi.lib().sph_ns_find_neighbors_noalloc(xd, n, radius, od, nd, capacity, C.byref(total), None)
        off = hip.get(od, np.zeros(n + 1, np.uint32))
        idx = hip.get(nd, np.zeros(total.value if rc == 0 else 0, np.uint32))
    finally:
        hip.free(xd, od, nd)
    return rc, total.value, off, idx


@pytest.mark.parametrize("seed", [0])
def test_noalloc_equals_drop_in_on_two_calls(seed):
    radius = 0.02
    for n in (60_000, 7_000):  # second call smaller than the first
        x = cloud(n, seed + n)
        print(f"noalloc: {n} points, radius {radius}", flush=True)
        off_r, idx_r = drop_in(x, radius)
        total_r = int(off_r[-1])
        rc, total, off, idx = noalloc(x, radius, total_r)
        assert rc == 0, capi.lib().sph_last_error().decode()
        assert total == total_r
        np.testing.assert_array_equal(off, off_r)
        np.testing.assert_array_equal(idx, idx_r)


def test_noalloc_capacity_and_limits():
    radius = 0.05
    x = cloud(20_000, 5)
    off_r, idx_r = drop_in(x, radius)
    total_r = int(off_r[-1])
    # too small: fails with the size needed, offsets already written
    rc, total, off, _ = noalloc(x, radius, total_r - 1)
    assert rc == SPH_ERR_RANGE and total == total_r
    np.testing.assert_array_equal(off, off_r)
    # retried with the reported size
    rc, total, off, idx = noalloc(x, radius, total)
    assert rc == 0
    np.testing.assert_array_equal(idx, idx_r)
    # an empty set
    rc, total, off, _ = noalloc(np.zeros((0, 3), np.float32), radius, 0)
    assert rc == 0 and total == 0 and off[0] == 0
    # beyond the maximum point count: refused before any device work
    total = C.c_size_t(7)
    rc = capi.lib().sph_ns_find_neighbors_noalloc(None, (1 << 19) + 1, radius, None, None, 0, C.byref(total), None)
    assert rc == SPH_ERR_RANGE
    assert "maximum" in capi.lib().sph_last_error().decode()


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_lists_at_any_output_alignment(shift):
    """Large sets are written in groups of four entries: the lists are whole
    and the words around them untouched at every alignment of the buffer."""
    n, radius = 131_200, 0.025
    x = np.random.default_rng(5).random((n, 3)).astype(np.float32)
    off_r, idx_r = drop_in(x, radius)
    hip = Hip()
    pad = 8
    xd, od, nd = hip.alloc(12 * n), hip.alloc(4 * (n + 1)), hip.alloc(4 * (len(idx_r) + 2 * pad))
    try:
        hip.put(xd, x.reshape(-1))
        hip.put(nd, np.full(len(idx_r) + 2 * pad, 0xABCDEF01, np.uint32))
        total = C.c_size_t(0)
        rc = capi.lib().sph_ns_find_neighbors_noalloc(xd, n, radius, od, C.c_void_p(nd.value + 4 * (pad - shift)),
                                                      len(idx_r), C.byref(total), None)
        off = hip.get(od, np.zeros(n + 1, np.uint32))
        buf = hip.get(nd, np.zeros(len(idx_r) + 2 * pad, np.uint32))
    finally:
        hip.free(xd, od, nd)
    assert rc == 0 and total.value == len(idx_r)
    np.testing.assert_array_equal(off, off_r)
    lo = pad - shift
    np.testing.assert_array_equal(buf[lo:lo + len(idx_r)], idx_r)
    assert (buf[:lo] == 0xABCDEF01).all() and (buf[lo + len(idx_r):] == 0xABCDEF01).all()
