"""Colliders of more candidates than a flat list holds (a large collider widens everyone's
query): from none to more contacts than the registers, and than the list, keep.
Bit for bit the oracle's, events included.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("n,squeeze,radius,mixed", [(250, 1.0, 3.0, False), (250, 0.4, 5.0, True), (900, 0.3, 4.0, False),
                                                    (900, 0.2, 6.0, True), (3000, 0.5, 9.0, False)])
def test_contacts_are_the_oracles(n, squeeze, radius, mixed):
    rng = np.random.default_rng(n)
    sc = scenes.plain_large_scene(n=2 * n, seed=9)
    middle = sc.pos.mean(0)
    sc.pos = ((sc.pos - middle) * squeeze + middle).astype(np.float32)
    # two centred colliders a body: no position depends on a rotation, whose last bits are libm's
    sc.col_parent = np.repeat(np.arange(2 * n), 2).astype(np.int32)
    m = len(sc.col_parent)
    sc.col_off = np.zeros((m, 2), np.float32)
    sc.col_abs = sc.pos[sc.col_parent].copy()
    sc.col_r = rng.uniform(0.2, 0.9, m).astype(np.float32)
    sc.col_r[7] = radius
    sc.col_mass_override, sc.col_has_mo = np.zeros(m, np.float32), np.zeros(m, np.uint8)
    sc.col_sensor = (rng.random(m) < 0.1).astype(np.uint8) if mixed else np.zeros(m, np.uint8)
    pick = (lambda: rng.integers(1, 4, m)) if mixed else (lambda: np.full(m, 0xFFFFFFFF))
    sc.col_mem, sc.col_filt = pick().astype(np.uint32), pick().astype(np.uint32)
    p = sc.build_physics()[0]
    p.set_event_capacity(1 << 20)
    o = OracleWorld(sc, np.float32, event_cap=1 << 20)
    for _ in range(2):
        p.step(sc.dt)
        o.step(sc.dt, 1)
        got = p.bodies()
        assert np.array_equal(bits(got["position"]), bits(o.pos))
        assert np.array_equal(bits(got["velocity"]), bits(o.vel))
    assert p.contact_count() == o.contact_count
    hs, vs, dropped = p.drain_events()
    cols, vels = o.events
    assert dropped == 0 and np.array_equal((hs & np.uint64(0xFFFFFFFF)).astype(np.int64), cols.astype(np.int64))
    assert np.array_equal(bits(vs), bits(vels))
