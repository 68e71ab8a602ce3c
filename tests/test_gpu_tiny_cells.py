"""Grids fitted to bodies whose radii and distances are a few of the least floats,
where a cell size times a little more than one is the same cell size: the fit
ends, and results are the oracle's and the same on every path.  So for a box too
wide for the type.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import Physics
from blobs_amd.rollout import Rollout
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu
LEAST = np.float32(1.4e-45)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def tiny(n, radius, width):
    """n bodies with radii and a box in units of the least float."""
    sc = scenes.plain_large_scene(n=n, seed=3)
    rng = np.random.default_rng(n)
    sc.pos = (rng.integers(0, width, (n, 2)).astype(np.float32) * LEAST).astype(np.float32)
    sc.pos[0], sc.pos[-1] = 0.0, np.float32(width) * LEAST
    sc.col_abs = sc.pos[sc.col_parent].copy()
    sc.col_r = np.full(n, np.float32(radius) * LEAST, np.float32)
    sc.vreq = np.zeros((n, 2), np.float32)
    sc.gravity = (0.0, 0.0)
    return sc


CASES = [(1, 200), (1, 3000), (2, 700), (3, 20000), (4, 1000), (6, 300)]


@pytest.mark.parametrize("radius,width", CASES)
@pytest.mark.parametrize("n", [12, 60])
def test_tiny_world_is_the_oracles(n, radius, width):
    sc = tiny(n, radius, width)  # (on the general path: its bodies coincide)
    p, o = sc.build_physics()[0], OracleWorld(sc, np.float32)
    for _ in range(2):
        p.step(sc.dt)
        o.step(sc.dt, 1)
        assert np.array_equal(bits(p.bodies()["position"]), bits(o.pos))


@pytest.mark.parametrize("radius,width", CASES)
def test_tiny_worlds_of_a_batch_and_a_rollout(radius, width):
    scs = [tiny(n, radius, width) for n in (5, 24)]
    made = [[sc.build_physics()[0] for sc in scs] for _ in range(3)]
    a, b = Physics.batch(made[0]), Physics.batch(made[1])
    b.set_broadphase(1.25, 1, 0.25)
    r = Rollout(made[2], np.zeros((2, 2), np.float32), checkpoint_every=1)
    for w in (a, b):
        w.step(scs[0].dt, 2)
    r.forward(scs[0].dt, 2)
    assert np.array_equal(bits(a.bodies()["position"]), bits(b.bodies()["position"]))
    assert np.array_equal(bits(a.bodies()["position"]), bits(r.final_positions()))


@pytest.mark.parametrize("persistent", [False, True])
def test_world_wider_than_the_type(persistent):
    """Two bodies so far apart that their distance overflows: the box is cut to the type's range."""
    scs = [scenes.plain_large_scene(n=n, seed=5) for n in (1100, 30)]
    for sc in scs:
        sc.pos[3], sc.pos[7] = (3e38, -3e38), (-3e38, 3e38)
        sc.col_abs = sc.pos[sc.col_parent].copy()
    b = Physics.batch([sc.build_physics()[0] for sc in scs])
    b.set_persistent(persistent)
    b.step(scs[0].dt, 2)
    assert b.persistent_active() == persistent
    got, at = b.bodies()["position"], 0
    for sc in scs:
        o = OracleWorld(sc, np.float32)
        o.step(sc.dt, 2)
        assert np.array_equal(bits(got[at:at + len(sc.pos)]), bits(o.pos))
        at += len(sc.pos)
