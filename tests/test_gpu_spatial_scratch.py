"""The scratch of a SpatialHash query, one block or two (spatial.hip): the same hits on both sides of the
sizes where that changes as with the array that needs no allocation, and no jump in what a call costs.

The cost: beside its kernels a call of 30,000 points takes one allocation of at most 2 MiB and its release, one of
36,000 takes two, so at most twice as much; half as much again is allowed for the clock.
"""
import ctypes as C
import time

import numpy as np
import pytest

from blobs_amd import _lib as L
from blobs_amd.spatial import HIT, POINT, QUERY
from tests.devbuf import DevBuf

pytestmark = pytest.mark.gpu


class Case:
    def __init__(self, n, nq):
        rng = np.random.default_rng(n + nq)
        side = np.sqrt(n) * 1.2
        pts, qs = np.zeros(n, POINT), np.zeros(nq, QUERY)
        pts["position"] = rng.random((n, 2)) * side
        pts["radius"], pts["id"] = 0.5, np.arange(n)
        pts["cell"] = np.floor(pts["position"] / 2.0).astype(np.int32)
        qs["position"] = rng.random((nq, 2)) * side
        qs["radius"] = 1.0
        self.lib, self.n, self.nq, self.cap = L.load(), n, nq, 16 * nq
        self.pts, self.qs = DevBuf(self.lib, pts.nbytes, pts), DevBuf(self.lib, qs.nbytes, qs)
        self.off, self.hits = DevBuf(self.lib, 4 * (nq + 1)), DevBuf(self.lib, HIT.itemsize * self.cap)

    def call(self, fn):
        total = C.c_uint64()
        L.check(fn(2.0, self.pts.p, self.n, self.qs.p, self.nq, self.off.p, self.hits.p, self.cap, C.byref(total)), None)
        return total.value

    def result(self, fn):
        n = self.call(fn)
        return self.off.get(np.uint32, self.nq + 1), self.hits.get(HIT, n)


@pytest.mark.parametrize("n,nq", [(18_000, 500), (19_000, 500), (32_768, 100), (32_769, 100), (40_000, 45_000),
                                  (65_536, 1000), (65_537, 1000)])
def test_same_hits_as_without_an_allocation(n, nq):
    c = Case(n, nq)
    a, b = c.result(c.lib.bg_spatial_hash_query), c.result(c.lib.bg_spatial_hash_query_noalloc)
    assert len(a[1]) > nq
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


def test_cost_of_the_scratch_has_no_jump():
    def cost(n):
        c = Case(n, 1000)
        fns = c.lib.bg_spatial_hash_query, c.lib.bg_spatial_hash_query_noalloc
        times = [], []
        for _ in range(80):
            for fn, t in zip(fns, times):
                t0 = time.perf_counter()
                c.call(fn)
                t.append(time.perf_counter() - t0)
        with_, without = (np.median(t) for t in times)
        return with_ - without

    assert cost(36_000) < 3.0 * cost(30_000)
