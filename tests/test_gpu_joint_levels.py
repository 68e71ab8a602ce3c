"""The joint stage by levels (k_joints): groups of components swept by one
workgroup each, staged in LDS or not, and rotation steps evaluated per solve.
Bodies carry one centred collider, so positions do not depend on rotations:
positions are the oracle's bit for bit; a rotation step is corr * h with corr
from a pair of f64 atan2 rounded to f32, so two libraries' may differ in the
last bit of an angle (2^-22 below pi) each.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def scene(kind, n=700):
    sc = scenes.plain_large_scene(n=n, seed=21)
    rng = np.random.default_rng(5)
    if kind == "pairs":
        a, b = np.arange(0, 400, 2), np.arange(1, 400, 2)
    elif kind == "chain":  # a component past every LDS table
        a, b = np.arange(0, 330), np.arange(1, 331)
    elif kind == "star":  # one solve a level
        a, b = np.zeros(100, int), np.arange(1, 101)
    elif kind == "ragged":  # components of 1 to 90 joints, some about the size of a group
        sizes = [1, 62, 2, 63, 64, 65, 1, 90, 5]
        a, b, at = [], [], 0
        for s in sizes:
            a += list(range(at, at + s))
            b += list(range(at + 1, at + s + 1))
            at += s + 1
        a, b = np.array(a), np.array(b)
    else:  # "mixed": random pairs, statics, anchors, some of them coincident
        a = rng.integers(0, n, 300)
        b = (a + 1 + rng.integers(0, n - 1, 300)) % n
        sc.body_type = sc.body_type.copy()
        sc.body_type[rng.integers(0, n, 60)] = 1
    sc.joint_a, sc.joint_b = a.astype(np.int32), b.astype(np.int32)
    sc.joint_anchor_a = np.zeros((len(a), 2), np.float32)
    sc.joint_anchor_b = np.zeros((len(a), 2), np.float32)
    if kind == "mixed":
        sc.joint_anchor_a = rng.normal(size=(300, 2)).astype(np.float32)
        sc.joint_anchor_a[:40] = sc.pos[b[:40]] - sc.pos[a[:40]]
    return sc


@pytest.mark.parametrize("kind", ["pairs", "chain", "star", "ragged", "mixed"])
@pytest.mark.parametrize("iterations", [(4,), (1, 7, 0, 4)])
def test_joint_sweep_is_the_sequential_one(kind, iterations):
    sc = scene(kind)
    p = sc.build_physics()[0]
    o = OracleWorld(sc, np.float32)
    turns = 0
    for it in iterations:
        p.joint_iterations = it
        o.w.joint_iterations = it
        p.step(sc.dt, 2)
        o.step(sc.dt, 2)
        turns += 2 * 8 * it * 100
        got = p.bodies()
        assert np.array_equal(bits(got["position"]), bits(o.pos))
        assert np.array_equal(bits(got["velocity"]), bits(o.vel))
        # at most 100 joints a body; each step's angle error is two last bits, times h, and the
        # sum's own rounding (rotations stay below 2^4 here)
        tol = turns * (2.0 ** -21 * sc.dt / 8 + 2.0 ** -20)
        assert np.abs(np.asarray(got["rotation"], np.float64) - np.asarray(o.rot, np.float64)).max() <= tol
    assert np.abs(o.rot).max() > 0
