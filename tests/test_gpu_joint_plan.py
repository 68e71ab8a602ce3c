"""The joints' schedule is kept across uploads that change nothing of it, and made
anew for changed joints, static bodies and iterations.
"""
import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import STATIC

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("n,joints", [(40, 12), (400, 150), (300, 700)])
def test_uploads_between_steps(n, joints):
    sc = scenes.multi_collider_scene(n=n, n_springs=n // 4, n_joints=joints, seed=8)
    (a, ha), (b, hb) = sc.build_physics(), sc.build_physics()

    def steps(k, reload):
        for _ in range(k):
            if reload:  # each step of `a` after an upload; `b` goes up only where something changed
                a.set_rbd(int(ha[0]), a.get_rbd(int(ha[0])))
            a.step(sc.dt)
            b.step(sc.dt)
        x, y = a.bodies(), b.bodies()
        for f in ("position", "velocity", "rotation"):
            assert np.array_equal(np.isnan(x[f]), np.isnan(y[f]))
            assert np.array_equal(bits(np.nan_to_num(x[f])), bits(np.nan_to_num(y[f]))), f

    steps(4, True)
    for w in (a, b):
        w.joint_iterations = 2
    steps(3, True)
    for w, h in ((a, ha), (b, hb)):
        r = w.get_rbd(int(h[sc.joint_a[0]]))
        r.body_type = STATIC
        w.set_rbd(int(h[sc.joint_a[0]]), r)
    steps(3, True)
    for w, h in ((a, ha), (b, hb)):
        w.create_fixed_joint(int(h[1]), int(h[n - 1]), (0.1, 0.0), (0.0, 0.1))
    steps(3, True)
    for w in (a, b):
        w.joint_iterations = 0
    steps(2, False)
    for w in (a, b):
        w.joint_iterations = 4
    steps(2, True)
