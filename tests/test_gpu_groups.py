"""A part of a scene far off as a group: the box of the grid is cut to the spread of
the bodies, and one that lies wholly outside would crowd a cell at its corner.
"""
import time

import numpy as np
import pytest

from blobs_amd import scenes

pytestmark = pytest.mark.gpu


def parted(sc, share, by):
    """The rightmost `share` of the bodies moved off by (by, by)."""
    far = np.zeros(len(sc.pos), bool)
    far[np.argsort(sc.pos[:, 0])[int(len(far) * (1 - share)):]] = True
    shift = np.where(far[:, None], np.float32(by), np.float32(0.0)).astype(np.float32) * np.ones((1, 2), np.float32)
    sc.pos = (sc.pos + shift).astype(np.float32)
    sc.col_abs = (sc.col_abs + shift[sc.col_parent]).astype(np.float32)
    return sc


def took(sc, before):
    p = sc.build_physics()[0]
    p.step(sc.dt, before)
    t = time.perf_counter()
    p.step(sc.dt, 4)
    return time.perf_counter() - t


def plain():
    return scenes.plain_large_scene(n=50021, seed=5)


def multi():
    return scenes.multi_collider_scene(n=32768, n_springs=0, n_joints=0, seed=5)


@pytest.mark.parametrize("make,share", [(plain, 0.07), (plain, 0.08), (multi, 0.01), (multi, 0.07)])
@pytest.mark.parametrize("before", [2, 12])
def test_a_group_far_off_crowds_no_cell(make, share, before):
    apart, together = took(parted(make(), share, 5000.0), before), took(make(), before)
    assert apart < 5.0 * together


@pytest.mark.parametrize("share", [0.01, 0.07])
def test_a_box_that_is_clipped_again(share):
    """Past the substeps after an upload, and past a hold: the whole box's bits."""
    scs = [parted(scenes.multi_collider_scene(n=2000, n_springs=0, n_joints=0, seed=5), share, 5000.0) for _ in range(2)]
    a, b = (sc.build_physics()[0] for sc in scs)
    h = int(b.bodies()["handles"][0])
    for _ in range(150):
        a.step(scs[0].dt)
        b.step(scs[0].dt)
        b.set_rbd(h, b.get_rbd(h))  # an upload, after which no box is clipped
    x, y = a.bodies(), b.bodies()
    for k in ("position", "velocity", "rotation"):
        assert np.array_equal(np.nan_to_num(x[k]), np.nan_to_num(y[k])), k
    assert a.contact_count() == b.contact_count()
