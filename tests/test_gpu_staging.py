"""The pinned memory of bulk reads: lent for one read, from a pool that outlives
worlds, so that the first read of a new world costs what a later one does; with
several threads at once; and with worlds of any size that come and go.
"""
import threading
import time

import numpy as np
import pytest

from blobs_amd import scenes

pytestmark = pytest.mark.gpu
FIELDS = ("position", "position_old", "velocity", "rotation", "angular_velocity")


def mirror(p):
    """The state through the host mirror."""
    p.get_rbd(int(p.bodies()["handles"][0]))
    return p.bodies()


def test_first_read_of_a_new_world():
    sc = scenes.plain_large_scene(n=600, seed=3)
    first, later, keep = [], [], []
    for _ in range(24):
        p = sc.build_physics()[0]
        keep.append(p)
        for out in (first, later):
            p.step(sc.dt)
            t = time.perf_counter()
            p.bodies()
            out.append(time.perf_counter() - t)
    assert np.median(first[4:]) < 2.5 * np.median(later[4:])


def test_reads_of_several_threads():
    scs = [scenes.plain_large_scene(n=n, seed=n) for n in (50, 900, 7000, 20000, 60000, 3000)]
    wrong = []

    def work(sc):
        try:
            for _ in range(3):
                p = sc.build_physics()[0]
                for _ in range(4):
                    p.step(sc.dt)
                    b = p.bodies()
                    m = mirror(p)
                    if not all(np.array_equal(b[k], m[k]) for k in FIELDS):
                        wrong.append(sc.n_bodies)
        except Exception as e:  # noqa: BLE001
            wrong.append(e)

    threads = [threading.Thread(target=work, args=(sc,)) for sc in scs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_worlds_that_come_and_go():
    for n in (30, 100000, 400, 1200000, 5, 7282):
        sc = scenes.plain_large_scene(n=n, seed=2)
        p = sc.build_physics()[0]
        p.step(sc.dt)
        b, c = p.bodies(), p.collider_positions()
        m = mirror(p)
        assert all(np.array_equal(b[k], m[k]) for k in FIELDS)
        assert np.array_equal(c, p.collider_positions())
        del p
