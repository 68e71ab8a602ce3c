"""State read back in bulk straight from the device (bg_get_bodies,
bg_get_collider_positions after a step) against the host mirror that every
single-body getter fills: bit for bit, in arena order, for worlds whose state
goes through pinned memory in one store and for larger ones that come over in
pieces, on both step paths, with removed bodies, in batches, and for any
subset of the arrays.
"""
import ctypes as C

import numpy as np
import pytest

from blobs_amd import _lib as L
from blobs_amd import scenes
from blobs_amd.physics import Physics

pytestmark = pytest.mark.gpu
FIELDS = ("position", "position_old", "velocity", "rotation", "angular_velocity")


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def check(p, sample):
    b, c = p.bodies(), p.collider_positions()  # from the device
    p.get_rbd(int(b["handles"][0]))            # fills the host mirror
    for h in sample(b["handles"]):
        r = p.get_rbd(int(h))
        k = int(np.flatnonzero(b["handles"] == h)[0])
        assert np.array_equal(bits(r.position), bits(b["position"][k]))
        assert np.array_equal(bits(r.calculated_velocity), bits(b["velocity"][k]))
    m, mc = p.bodies(), p.collider_positions()  # from the host mirror
    for f in FIELDS:
        assert np.array_equal(bits(b[f]), bits(m[f])), f
    assert np.array_equal(b["handles"], m["handles"])
    assert np.array_equal(bits(c), bits(mc))


@pytest.mark.parametrize("kind,n", [("plain", 1), ("plain", 64), ("plain", 7281), ("plain", 7282), ("plain", 120000),
                                    ("multi", 48), ("multi", 9000)])
def test_read_back_equals_the_host_mirror(kind, n):
    if kind == "plain":
        sc = scenes.plain_large_scene(n=n, seed=7)
    else:
        sc = scenes.multi_collider_scene(n=n, n_springs=n // 2, n_joints=n // 4, seed=7)
    p, bh = sc.build_physics()
    p.step(sc.dt, 2)
    check(p, lambda h: h[:: max(1, len(h) // 20)])
    if kind == "plain" and n > 10:  # (a spring or joint of a removed body panics)
        p.remove_rbd(int(bh[3]))
        p.remove_rbd(int(bh[n - 1]))
        p.step(sc.dt, 1)
        check(p, lambda h: h[:: max(1, len(h) // 20)])


@pytest.mark.parametrize("sizes", [(64, 5, 300), (5000, 64, 9000)])
def test_batches_and_their_old_dt(sizes):
    rng = scenes.Rng(31)
    scs = [scenes.uneven_batch_world(n, 0.3, rng) for n in sizes]
    src = [sc.build_physics()[0] for sc in scs]
    b = Physics.batch(src)
    b.step(1 / 60, 2)
    got = b.bodies()
    b.writeback(src)
    lo = 0
    for sc, w in zip(scs, src):
        own = w.bodies()
        for f in FIELDS:
            assert np.array_equal(bits(got[f][lo:lo + sc.n_bodies]), bits(own[f])), f
        assert w.old_dt == pytest.approx(1 / 480)
        lo += sc.n_bodies


@pytest.mark.parametrize("n", [500, 20000])
def test_any_subset_of_the_arrays(n):
    sc = scenes.plain_large_scene(n=n, seed=9)
    p, _ = sc.build_physics()
    p.step(sc.dt, 2)
    full = p.bodies()
    p.step(sc.dt, 1)
    rot = np.zeros(n, np.float32)
    assert L.load().bg_get_bodies(p._w, None, None, None, L.fptr(rot), None, None) == L.BG_OK
    old = np.zeros((n, 2), np.float32)
    assert L.load().bg_get_bodies(p._w, None, L.fptr(old), None, None, None, None) == L.BG_OK
    assert p.old_dt == pytest.approx(1 / 960)  # brought along, as by a full read
    cnt = C.c_uint32()
    assert L.load().bg_get_collider_positions(p._w, None, C.byref(cnt)) == L.BG_OK and cnt.value == n
    after = p.bodies()
    assert np.array_equal(bits(rot), bits(after["rotation"]))
    assert np.array_equal(bits(old), bits(after["position_old"]))
    assert not np.array_equal(after["position"], full["position"])
