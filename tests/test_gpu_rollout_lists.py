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


@pytest.mark.parametrize("partners", [1, 2, 15, 16, 17, 18, 33, 1500])
@pytest.mark.parametrize("n", [256, 700, 2048])
def test_bodies_of_many_partners_in_rounds(n, partners):
    """Hubs with so many bodies touching them and no others, in random index order; more pairs than the
    queue holds at once, where a body's last 16 partners are kept from the walk that counts them, and
    a hub of more than the queue ever holds (1,200 pairs, worlds past 1,024 bodies)."""
    rng = np.random.default_rng(n + partners)
    sc = scenes.rollout_world(n, 8, scenes.Rng(42), damping=1.0)
    size = partners + 1
    k = np.arange(n)
    hub, member = k // size, k % size
    wide = int(np.ceil(np.sqrt(n / size)))
    at = np.stack([hub % wide, hub // wide], 1) * 12.0 - 6.0 * wide
    angle = 2.0 * np.pi * member / max(partners, 1)
    at += np.where(member[:, None] > 0, 4.0 * np.stack([np.cos(angle), np.sin(angle)], 1), 0.0)
    order = rng.permutation(n)
    sc.pos, sc.col_r = np.zeros((n, 2), np.float32), np.zeros(n, np.float32)
    sc.pos[order] = at + rng.uniform(-0.02, 0.02, (n, 2))
    sc.col_r[order] = np.where(member > 0, 0.33, 3.75)
    sc.col_abs = sc.pos.copy()
    got = [run([sc], 3, ck) for ck in (1, 2)]
    o = OracleWorld(sc, np.float32)
    o.step(sc.dt, 3)
    assert np.array_equal(bits(got[0][0]), bits(o.pos))
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))


@pytest.mark.parametrize("n", [200, 321, 700, 1300, 2048])
def test_a_body_over_all_others(n):
    """One body outside the lists and in contact with everyone, who touch nobody else: as many pairs as the
    queue still holds, and more than it ever does (past 1,200)."""
    rng = np.random.default_rng(n)
    sc = scenes.rollout_world(n, 8, scenes.Rng(43), damping=1.0)
    wide = int(np.ceil(np.sqrt(n)))
    k = np.arange(n)
    at = np.stack([k % wide, k // wide], 1) * 2.5 - 1.25 * wide + rng.uniform(-0.2, 0.2, (n, 2))
    order = rng.permutation(n)
    sc.pos, sc.col_r = np.zeros((n, 2), np.float32), np.zeros(n, np.float32)
    sc.pos[order] = at
    sc.col_r[order] = 0.5
    sc.pos[n // 3], sc.col_r[n // 3] = (0.3, -0.2), 2.0 * wide
    sc.col_abs = sc.pos.copy()
    got = [run([sc], 3, ck) for ck in (1, 2)]
    o = OracleWorld(sc, np.float32)
    o.step(sc.dt, 3)
    assert np.array_equal(bits(got[0][0]), bits(o.pos))
    for a, b in zip(*got):
        assert np.array_equal(bits(a), bits(b))
