"""Small worlds (small_kernels.hip) past what their lists and counters hold: with
bodies of more partners than a list they stay on their path, through chunks of
any length, with the grid path's bits; and chunks of any number of steps run all
of them.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import Physics

pytestmark = pytest.mark.gpu

GRID = (1.25, 1, 0.25)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def crowd(n, seed=5):
    sc = scenes.plain_large_scene(n=n, seed=seed)
    sc.pos = (np.random.default_rng(seed + n).random((n, 2)) * 0.25 * np.sqrt(n)).astype(np.float32)
    return sc


@pytest.mark.parametrize("chunk,chunks", [(3, 3), (1, 5), (5, 2)])
@pytest.mark.parametrize("sizes", [(300,), (90, 300, 40)])
def test_chunks_of_overflowing_worlds(sizes, chunk, chunks):
    # past 256 steps, at each call: a tail that is captured to follow replayed graphs takes their path
    scs = [crowd(n) for n in sizes]
    made = [[sc.build_physics()[0] for sc in scs] for _ in range(2)]
    a, b = (ws[0] if len(ws) == 1 else Physics.batch(ws) for ws in made)
    b.set_broadphase(*GRID)
    for call in range(320 // (chunk * chunks)):
        for w in (a, b):
            w.run_chunks(scs[0].dt, chunk, chunks)
        sa, sb = a.bodies(), b.bodies()
        for k in ("position", "position_old", "velocity", "rotation"):
            assert np.array_equal(bits(sa[k]), bits(sb[k])), (k, call)
    assert a.contact_count() == b.contact_count() > 0


def test_chunks_of_more_than_32_bits_of_steps():
    """(Of no substeps each, so that only the clock moves.)"""
    p = crowd(20).build_physics()[0]
    p.substeps = 0
    p.run_chunks(2.0 ** -20, 1 << 16, 1 << 16)
    assert p.time == 2.0 ** 12
