"""The rollout kernels at the edges of their workgroup: one, two and 1,024 or
1,025 bodies (one or two a thread), worlds with as many springs or joints as
LDS holds and with one more, bodies of more springs than a thread packs, and
recomputes of one or of several segments a launch.

Bars: final positions bit-exact against the oracle; gradients equal, value by
value, for every checkpoint interval; and a world with one spring of zero
stiffness, or one joint between two bodies nobody else touches, more than LDS
holds (which moves it to the other path) has the other bodies' and springs'
very gradients.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.rollout import Rollout
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def world(n, springs, joints=0, seed=90, damping=2.0):
    rng = scenes.Rng(seed)
    return scenes.rollout_world(n, springs, rng, damping=damping if springs else 0.0, n_joints=joints,
                                anchor=0.2 if joints else 0.0)


def run(ws, steps, ck):
    r = Rollout([w.build_physics()[0] for w in ws], np.zeros((len(ws), 2), np.float32), checkpoint_every=ck)
    r.forward(ws[0].dt, steps)
    pos = r.final_positions()
    gv, gk = r.backward()
    return pos, gv, gk


@pytest.mark.parametrize("n,springs,joints", [(1, 0, 0), (2, 1, 0), (65, 200, 0), (1024, 100, 20), (1025, 2048, 0),
                                              (700, 2049, 30), (2048, 1024, 0), (900, 0, 256), (900, 10, 257)])
def test_forward_matches_the_oracle_and_gradients_the_interval(n, springs, joints):
    ws = [world(n, springs, joints), world(max(n // 3, 2), min(springs, 5), min(joints, 1), seed=91)]
    steps = 5
    got = [run(ws, steps, ck) for ck in (1, 2, 5)]
    b0 = 0
    for sc in ws:
        o = OracleWorld(sc, np.float32)
        o.step(sc.dt, steps)
        assert np.array_equal(bits(got[0][0][b0:b0 + sc.n_bodies]), bits(o.pos))
        b0 += sc.n_bodies
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(bits(a), bits(b))
    assert np.isfinite(got[0][1]).all() and np.abs(got[0][1]).max() > 0


def test_one_spring_more_than_lds_holds():
    a, b = world(600, 2048), world(600, 2048)
    b.spring_a = np.append(b.spring_a, np.int32(0))
    b.spring_b = np.append(b.spring_b, np.int32(1))
    b.spring_rest = np.append(b.spring_rest, np.float32(1.0))
    b.spring_k = np.append(b.spring_k, np.float32(0.0))
    b.spring_c = np.append(b.spring_c, np.float32(0.0))
    (pa, va, ka), (pb, vb, kb) = run([a], 4, 2), run([b], 4, 2)
    assert np.array_equal(pa, pb)
    assert np.array_equal(va, vb)
    assert np.array_equal(ka, kb[:2048])


def test_one_joint_more_than_lds_holds():
    a, b = world(800, 50, 256), world(800, 50, 256)
    for sc in (a, b):  # two bodies far from everyone, moving like nobody else
        for arr in (sc.pos, sc.col_abs):
            arr[-2:] = [(300.0, 300.0), (303.0, 300.0)]
        keep = ~(np.isin(sc.joint_a, (798, 799)) | np.isin(sc.joint_b, (798, 799)))
        first = np.flatnonzero(keep)[0]
        sc.joint_a[~keep], sc.joint_b[~keep] = sc.joint_a[first], sc.joint_b[first]
        on = np.isin(sc.spring_a, (798, 799)) | np.isin(sc.spring_b, (798, 799))
        sc.spring_a[on], sc.spring_b[on] = 0, 1
    b.joint_a = np.append(b.joint_a, np.int32(798))
    b.joint_b = np.append(b.joint_b, np.int32(799))
    b.joint_anchor_a = np.vstack([b.joint_anchor_a, np.zeros((1, 2), np.float32)])
    b.joint_anchor_b = np.vstack([b.joint_anchor_b, np.zeros((1, 2), np.float32)])
    dl = np.zeros((800, 2), np.float32)  # a loss the two have no part in
    dl[:798] = np.random.default_rng(5).normal(size=(798, 2))
    out = []
    for sc in (a, b):
        r = Rollout([sc.build_physics()[0]], np.zeros((1, 2), np.float32), checkpoint_every=2)
        r.forward(sc.dt, 4)
        out.append((r.final_positions(), *r.backward(dl)))
    (pa, va, ka), (pb, vb, kb) = out
    assert np.array_equal(pa[:798], pb[:798])
    assert np.array_equal(va[:798], vb[:798])
    assert np.array_equal(ka, kb)
