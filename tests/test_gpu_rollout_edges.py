"""Rollouts at the edges of their parameters."""
import ctypes as C

import numpy as np
import pytest

from blobs_amd import _lib as L
from blobs_amd import scenes
from blobs_amd.rollout import Rollout
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def free_memory():
    """Of the card, by the HIP runtime that the library itself runs on (torch's is another one)."""
    free, total = C.c_size_t(), C.c_size_t()
    assert L.load().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("joints", [0, 5])
def test_worlds_of_no_substeps(joints):
    """Nothing moves, and no parameter has a gradient (a backward divided by the segment's substeps)."""
    sc = scenes.rollout_world(40, 20, scenes.Rng(3), damping=1.0, n_joints=joints, anchor=0.2)
    worlds = [sc.build_physics()[0] for _ in range(2)]
    for w in worlds:
        w.substeps = 0
    r = Rollout(worlds, np.zeros((2, 2), np.float32), checkpoint_every=2)
    loss = r.forward(sc.dt, 5)
    assert np.isfinite(loss).all()
    assert np.array_equal(r.final_positions(), np.concatenate([sc.pos, sc.pos]).astype(np.float32))
    gv, gk = r.backward()
    assert not gv.any() and not gk.any()


@pytest.mark.parametrize("every", [1, 2])
def test_memory_of_a_backward(every):
    """A backward takes at most 64 MiB beside the segment of tape that checkpoint_every stands for."""
    rng = scenes.Rng(4)
    scs = [scenes.rollout_world(2048, 0, rng) for _ in range(48)]
    r = Rollout([sc.build_physics()[0] for sc in scs], np.zeros((48, 2), np.float32), checkpoint_every=every)
    r.forward(scs[0].dt, 8)
    before = free_memory()
    gv, _ = r.backward()
    assert before - free_memory() <= 64 << 20
    assert np.isfinite(gv).all() and gv.any()


@pytest.mark.parametrize("joints", [4, 256, 257])  # staged in LDS, and one more than it holds
def test_joints_of_static_bodies(joints):
    """Every second joint holds its body a or b, or both, in place (the records carry the flags)."""
    sc = scenes.rollout_world(300, 20, scenes.Rng(9), damping=1.0, n_joints=joints, anchor=0.2)
    sc.body_type = sc.body_type.copy()
    sc.body_type[sc.joint_a[::4]] = 1
    sc.body_type[sc.joint_b[2::4]] = 1
    got = []
    for every in (1, 3):
        r = Rollout([sc.build_physics()[0]], np.zeros((1, 2), np.float32), checkpoint_every=every)
        r.forward(sc.dt, 4)
        got.append((r.final_positions(), *r.backward()))
    o = OracleWorld(sc, np.float32)
    o.step(sc.dt, 4)
    assert np.array_equal(got[0][0].view(np.uint32), np.ascontiguousarray(o.pos, np.float32).view(np.uint32))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
