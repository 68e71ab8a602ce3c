"""The cell grid of worlds whose box has more cells than their table: square and
thin boxes, boxes just past it, most bodies in a crowded middle.  Bit for bit
the oracle's, on the general path, as a plain world and in a batch.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import Physics
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def spread(sc, width, height, share, seed):
    """`share` of the bodies thrown into a box of the given size about the scene's middle."""
    rng = np.random.default_rng(seed)
    n = len(sc.pos)
    far = rng.random(n) < share
    box = (rng.random((n, 2)) - 0.5) * np.array([width, height])
    shift = np.where(far[:, None], box, 0.0).astype(np.float32)
    sc.pos = (sc.pos + shift).astype(np.float32)
    sc.col_abs = (sc.col_abs + shift[sc.col_parent]).astype(np.float32)
    return sc


def check(p, sc, steps):
    o = OracleWorld(sc, np.float32)
    p.step(sc.dt, steps)
    o.step(sc.dt, steps)
    got = p.bodies()
    assert np.array_equal(bits(got["position"]), bits(o.pos))
    assert np.array_equal(bits(got["velocity"]), bits(o.vel))
    assert p.contact_count() == o.contact_count


BOXES = [(300.0, 300.0, 0.3), (700.0, 700.0, 0.6), (30000.0, 20000.0, 0.5), (1.0e5, 2.0, 0.3), (0.0, 5.0e4, 0.3)]


@pytest.mark.parametrize("width,height,share", BOXES)
@pytest.mark.parametrize("n", [400, 1200])
def test_spread_general_world(width, height, share, n):
    sc = scenes.multi_collider_scene(n=n, n_springs=0, n_joints=0, seed=5)
    sc = spread(sc, width, height, share, 6)
    check(sc.build_physics()[0], sc, 3)


@pytest.mark.parametrize("width,height,share", BOXES)
def test_spread_plain_world(width, height, share):
    sc = spread(scenes.plain_large_scene(n=3000, seed=7), width, height, share, 8)
    check(sc.build_physics()[0], sc, 4)


def test_spread_worlds_of_a_batch():
    scs = [spread(scenes.plain_large_scene(n=n, seed=n), w, h, s, n) for n, (w, h, s) in zip((2100, 300, 2500, 900, 64), BOXES)]
    b = Physics.batch([sc.build_physics()[0] for sc in scs])
    b.step(scs[0].dt, 4)
    got, at = b.bodies()["position"], 0
    for sc in scs:
        o = OracleWorld(sc, np.float32)
        o.step(sc.dt, 4)
        assert np.array_equal(bits(got[at:at + len(sc.pos)]), bits(o.pos))
        at += len(sc.pos)
