"""Contacts of the general path: the wave's queue of pairs, its overflow (every
collider with many contacts), bodies of more colliders than merge lanes, and
colliders past their list -- each against the oracle bit for bit.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def scene(n, cols, side, rmax, seed, ragged=False, mixed=False):
    """n bodies of `cols` colliders (1 to cols when ragged) thrown into a square box."""
    rng = np.random.default_rng(seed)
    sc = scenes.multi_collider_scene(n=n, n_springs=0, n_joints=0, seed=seed)
    sc.pos = (rng.random((n, 2)) * side).astype(np.float32)
    count = rng.integers(1, cols + 1, n) if ragged else np.full(n, cols)
    parent = np.repeat(np.arange(n, dtype=np.int32), count)
    nc = len(parent)
    off = (rng.normal(size=(nc, 2)) * rmax).astype(np.float32)
    sc.col_parent, sc.col_off = parent, off
    sc.col_abs = (sc.pos[parent] + off).astype(np.float32)
    sc.col_r = (rmax * (0.3 + 0.7 * rng.random(nc))).astype(np.float32)
    sc.col_mass_override, sc.col_has_mo = np.zeros(nc, np.float32), np.zeros(nc, np.uint8)
    sc.col_sensor = (rng.random(nc) < 0.2).astype(np.uint8) if mixed else np.zeros(nc, np.uint8)
    sc.col_mem = (rng.integers(1, 4, nc) if mixed else np.full(nc, 0xFFFFFFFF)).astype(np.uint32)
    sc.col_filt = (rng.integers(1, 4, nc) if mixed else np.full(nc, 0xFFFFFFFF)).astype(np.uint32)
    return sc


@pytest.mark.parametrize("n,cols,side,ragged,mixed", [
    (40, 1, 40.0, False, True),  # no contacts
    (63, 2, 10.0, False, False),
    (64, 8, 30.0, True, False),
    (65, 9, 30.0, False, False),  # more colliders than merge lanes
    (200, 5, 14.0, True, True),  # the queue overflows
    (150, 12, 9.0, True, False),  # ... and lists too: bodies walked whole
    (700, 3, 60.0, True, True),
])
def test_contacts_are_the_oracles(n, cols, side, ragged, mixed):
    sc = scene(n, cols, side, 0.5, 3 * n + cols, ragged, mixed)
    p = sc.build_physics()[0]
    o = OracleWorld(sc, np.float32)
    for steps in (1, 2):
        p.step(sc.dt, steps)
        o.step(sc.dt, steps)
        got = p.bodies()
        assert np.array_equal(bits(got["position"]), bits(o.pos))
        assert np.array_equal(bits(got["velocity"]), bits(o.vel))
        assert p.contact_count() == o.contact_count
