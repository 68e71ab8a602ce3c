"""Small worlds (small_kernels.hip) past what their lists and counters hold: with
bodies of more partners than a list they stay on their path, through chunks of
any length, with the grid path's bits and in less than its time; and chunks of
any number of steps run all of them.
"""
import time

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


def pebbles(n, seed=5):
    """A large body among small ones, in a round container."""
    sc = scenes.plain_large_scene(n=n, seed=seed)
    lo, hi = sc.pos.min(0), sc.pos.max(0)
    sc.col_r[n // 2] = 4.0
    sc.con_pos = ((lo + hi) / 2).astype(np.float32)[None, :]
    sc.con_r = np.array([0.5 * float((hi - lo).max())], np.float32)
    return sc


def giant(n, seed=5):
    """One body that covers many others, with ragged radii."""
    sc = scenes.plain_large_scene(n=n, seed=seed)
    sc.col_r = (0.1 + 0.4 * np.random.default_rng(seed + n).random(n)).astype(np.float32)
    sc.col_r[n // 2] = 12.0
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


@pytest.mark.parametrize("make,n", [(pebbles, 300), (pebbles, 1000), (giant, 2000)])
def test_overflowing_world_takes_less_than_the_grid_path(make, n):
    # (in calls of thirty steps and in calls of one, after lists have overflowed)
    sc = make(n)
    a, b = sc.build_physics()[0], sc.build_physics()[0]
    b.set_broadphase(*GRID)
    took = {}
    for w in (a, b):
        w.step(sc.dt, 2)
        t0 = time.perf_counter()
        for _ in range(12):
            w.step(sc.dt)
        t1 = time.perf_counter()
        w.step(sc.dt, 30)
        took[w] = (t1 - t0, time.perf_counter() - t1)
    assert took[a][0] < 0.9 * took[b][0] and took[a][1] < 0.9 * took[b][1], list(took.values())
    assert np.array_equal(bits(a.bodies()["position"]), bits(b.bodies()["position"]))


def test_chunks_of_more_than_32_bits_of_steps():
    """(Of no substeps each, so that only the clock moves.)"""
    p = crowd(20).build_physics()[0]
    p.substeps = 0
    p.run_chunks(2.0 ** -20, 1 << 16, 1 << 16)
    assert p.time == 2.0 ** 12
