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


def took(sc):
    p = sc.build_physics()[0]
    p.step(sc.dt, 2)
    t = time.perf_counter()
    p.step(sc.dt, 4)
    return time.perf_counter() - t


def plain():
    return scenes.plain_large_scene(n=50021, seed=5)


@pytest.mark.parametrize("make,share", [(plain, 0.07), (plain, 0.08)])
def test_a_group_far_off_crowds_no_cell(make, share):
    apart, together = took(parted(make(), share, 5000.0)), took(make())
    assert apart < 5.0 * together
