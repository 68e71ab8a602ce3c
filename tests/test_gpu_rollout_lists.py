"""Rollouts whose contacts come from partner lists (diff_kernels.hip): at the
sizes where the workgroup changes, with bodies that leave their lists at once
(fast), worlds too dense for lists or for the queue of pairs (crowd, pile), and
a body among more partners than a list holds (giant).

Bars: final positions bit-exact against the oracle; gradients equal, value by
value, for checkpoint intervals whose recomputes start their lists elsewhere.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.rollout import Rollout
from oracle.oracle import OracleWorld

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def world(n, kind, seed):
    rng = np.random.default_rng(seed + n)
    sc = scenes.rollout_world(n, n // 2, scenes.Rng(seed), damping=1.0 if n > 1 else 0.0)
    if kind == "fast":
        sc.vreq = (rng.normal(size=(n, 2)) * 60.0).astype(np.float32)
    elif kind in ("crowd", "pile"):
        side = (0.35 if kind == "crowd" else 0.75) * np.sqrt(n)
        sc.pos = (rng.random((n, 2)) * side).astype(np.float32)
        sc.col_abs = sc.pos.copy()
    elif kind == "giant":
        sc.col_r = sc.col_r.copy()
        sc.col_r[n // 2] = 6.0
    return sc


def run(ws, steps, ck):
    r = Rollout([w.build_physics()[0] for w in ws], np.zeros((len(ws), 2), np.float32), checkpoint_every=ck)
    r.forward(ws[0].dt, steps)
    pos = r.final_positions()
    return (pos, *r.backward())


@pytest.mark.parametrize("kind", ["plain", "fast", "crowd", "pile", "giant"])
@pytest.mark.parametrize("n", [3, 64, 256, 257, 512, 513, 1024, 1025, 2048])
def test_lists_change_no_result(n, kind):
    ws = [world(n, kind, 40), world(max(n // 2, 2), "plain", 41)]
    steps = 4
    got = [run(ws, steps, ck) for ck in (1, 3)]
    b0 = 0
    for sc in ws:
        o = OracleWorld(sc, np.float32)
        o.step(sc.dt, steps)
        assert np.array_equal(bits(got[0][0][b0:b0 + sc.n_bodies]), bits(o.pos))
        b0 += sc.n_bodies
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))
