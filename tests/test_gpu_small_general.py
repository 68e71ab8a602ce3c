"""General-path worlds whose substep is four launches (k_small_contacts,
k_small_integrate), at and past the sizes where they take over: with springs,
joints, groups, sensors, events and push-outs, bit for bit against the oracle.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    """A spring between coincident bodies makes NaN, whose sign and payload are the processor's."""
    a = np.ascontiguousarray(a, np.float32)
    return np.where(np.isnan(a), np.uint32(0x7FC00000), a.view(np.uint32))


def scene(n, colliders, mixed=False, coincident=False, seed=3):
    """n bodies, `colliders` in all, the first of each centred and the rest on it (so that no
    position depends on a rotation, whose last bits are libm's)."""
    rng = np.random.default_rng(seed + n)
    sc = scenes.multi_collider_scene(n=n, n_springs=n // 2 if n > 1 else 0, n_joints=n // 4 if n > 3 else 0, seed=seed)
    extra = rng.integers(0, n, colliders - n)
    parent = np.sort(np.concatenate([np.arange(n), extra])).astype(np.int32)
    sc.col_parent = parent
    sc.col_off = np.zeros((colliders, 2), np.float32)
    sc.col_r = rng.uniform(0.2, 0.9, colliders).astype(np.float32)
    if coincident:
        sc.pos = sc.pos.copy()
        sc.pos[1] = sc.pos[0]
    sc.col_abs = sc.pos[parent].copy()
    sc.col_mass_override, sc.col_has_mo = np.zeros(colliders, np.float32), np.zeros(colliders, np.uint8)
    sc.col_sensor = (rng.random(colliders) < 0.2).astype(np.uint8) if mixed else np.zeros(colliders, np.uint8)
    pick = (lambda: rng.integers(1, 4, colliders)) if mixed else (lambda: np.full(colliders, 0xFFFFFFFF))
    sc.col_mem, sc.col_filt = pick().astype(np.uint32), pick().astype(np.uint32)
    return sc


@pytest.mark.parametrize("n,colliders,mixed,coincident", [
    (1, 2, False, False), (2, 3, False, True), (40, 63, True, False), (64, 64, False, False), (65, 128, False, False),
    (200, 1024, True, False), (250, 1151, False, False), (256, 1152, False, False), (256, 1153, False, False),
    (257, 1000, True, False), (100, 400, False, True),
])
def test_small_general_worlds_are_the_oracles(n, colliders, mixed, coincident):
    sc = scene(n, colliders, mixed, coincident)
    p = sc.build_physics()[0]
    p.set_event_capacity(1 << 16)
    o = OracleWorld(sc, np.float32, event_cap=1 << 16)
    for steps in (1, 3):
        p.step(sc.dt, steps)
        o.step(sc.dt, steps)
        got = p.bodies()
        assert np.array_equal(bits(got["position"]), bits(o.pos))
        assert np.array_equal(bits(got["velocity"]), bits(o.vel))
        assert p.contact_count() == o.contact_count
    hs, vs, dropped = p.drain_events()
    cols, vels = o.events
    assert dropped == 0
    assert np.array_equal((hs & np.uint64(0xFFFFFFFF)).astype(np.int64), cols.astype(np.int64))
    assert np.array_equal(bits(vs), bits(vels))
