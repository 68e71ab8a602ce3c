"""The rebuild interval a world chooses by itself (no bg_set_broadphase):
bodies so fast that most leave their skin within a step drive it down to
rebuilds inside a step, and a calm afterwards brings it up again.  Results are
the fixed interval's bit for bit, contacts included, and the oracle's.
"""
import time

import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import Physics
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def fast_scene(n, seed):
    sc = scenes.plain_large_scene(n=n, seed=seed)
    sc.vreq = (np.random.default_rng(seed).normal(size=(n, 2)) * 150.0).astype(np.float32)
    return sc


@pytest.mark.parametrize("n", [700, 6000, 70000])
@pytest.mark.parametrize("steps_per_call", [1, 3])
def test_adapted_interval_changes_no_result(n, steps_per_call):
    sc = fast_scene(n, 11)
    a, b = sc.build_physics()[0], sc.build_physics()[0]
    b.set_broadphase(1.25, 1, 0.25)
    for _ in range(9):
        a.step(sc.dt, steps_per_call)
        b.step(sc.dt, steps_per_call)
        assert np.array_equal(bits(a.bodies()["position"]), bits(b.bodies()["position"]))
    sa, sb = a.bodies(), b.bodies()
    for k in ("position_old", "velocity", "rotation"):
        assert np.array_equal(bits(sa[k]), bits(sb[k])), k
    assert a.contact_count() == b.contact_count() > 0


def test_adapted_interval_against_the_oracle():
    sc = fast_scene(5000, 12)
    p = sc.build_physics()[0]
    for _ in range(8):
        p.step(sc.dt)
    o = OracleWorld(sc, np.float32)
    o.step(sc.dt, 8)
    assert np.array_equal(bits(p.bodies()["position"]), bits(o.pos))
    assert np.array_equal(bits(p.bodies()["velocity"]), bits(o.vel))


def test_adapted_interval_of_a_batch_in_chunks():
    scs = [fast_scene(n, 20 + n) for n in (300, 2000, 5000)]
    a, b = (Physics.batch([sc.build_physics()[0] for sc in scs]) for _ in range(2))
    b.set_broadphase(1.5, 2, 0.25)
    for _ in range(6):
        a.run_chunks(scs[0].dt, 2, 3)
        b.run_chunks(scs[0].dt, 2, 3)
        assert np.array_equal(bits(a.bodies()["position"]), bits(b.bodies()["position"]))
    assert a.contact_count() == b.contact_count() > 0


@pytest.mark.parametrize("steps_per_call", [1, 40])
def test_adapted_interval_with_deferred_checks(steps_per_call):
    # one call's record is read while the next call, perhaps with a trial, is queued
    sc = fast_scene(3000, 13)
    a, b = sc.build_physics()[0], sc.build_physics()[0]
    a.set_deferred_checks(True)
    b.set_broadphase(1.25, 1, 0.25)
    for _ in range(240 // steps_per_call):
        a.step(sc.dt, steps_per_call)
        b.step(sc.dt, steps_per_call)
    a.synchronize()
    sa, sb = a.bodies(), b.bodies()
    for k in ("position", "position_old", "velocity"):
        assert np.array_equal(bits(sa[k]), bits(sb[k])), k


def test_outliers_by_thousands_leave_one_rebuild_a_step():
    """21,997 bodies of which 3,700 part from the rest: no slower than with one rebuild a step for good, a tenth
    allowed for the clock (with two a step 145 us against 121)."""
    sc = scenes.plain_large_scene(n=21997, seed=6)
    a, b = sc.build_physics()[0], sc.build_physics()[0]
    b.set_broadphase(1.25, 1, 0.25)
    t = [], []
    for call in range(30):
        for w, v in zip((a, b), t):
            w.bodies()
            t0 = time.perf_counter()
            w.step(sc.dt, 45)
            v.append(time.perf_counter() - t0)
    assert np.median(t[0][22:]) < 1.1 * np.median(t[1][22:])
    assert np.array_equal(bits(a.bodies()["position"]), bits(b.bodies()["position"]))
