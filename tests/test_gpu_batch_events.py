"""Events of small worlds whose buffer is too small: the ones kept are a prefix of
the reference's stream by whole substeps, and so the same on every path, for one
world and for several that record into one buffer.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import Physics

pytestmark = pytest.mark.gpu

GRID = (1.25, 1, 0.25)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def crowd(n, seed):
    sc = scenes.plain_large_scene(n=n, seed=seed)
    sc.pos = (np.random.default_rng(seed).random((n, 2)) * 0.8 * np.sqrt(n)).astype(np.float32)
    return sc


@pytest.mark.parametrize("sizes", [(700,), (40, 600, 90, 1300), tuple(range(20, 420, 3))])
@pytest.mark.parametrize("cap", [64, 1000, 20000])
@pytest.mark.parametrize("chunks", [False, True])
def test_kept_events_of_a_full_buffer(sizes, cap, chunks):
    scs = [crowd(n, 7 + n) for n in sizes]
    a, b = (Physics.batch([sc.build_physics()[0] for sc in scs]) if len(sizes) > 1 else scs[0].build_physics()[0]
            for _ in range(2))
    b.set_broadphase(*GRID)
    for w in (a, b):
        w.set_event_capacity(cap)
    for _ in range(2):
        for w in (a, b):
            if chunks:
                w.run_chunks(scs[0].dt, 2, 2)
            else:
                w.step(scs[0].dt, 3)
        (ha, va, da), (hb, vb, db) = a.drain_events(), b.drain_events()
        assert da == db
        assert np.array_equal(ha, hb) and np.array_equal(bits(va), bits(vb))
    assert a.contact_count() == b.contact_count()
