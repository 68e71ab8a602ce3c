"""Parameters set after a world's state was read in bulk (an export, which leaves the
host mirror behind) hold as after a read through the mirror.
"""
import numpy as np
import pytest

from blobs_amd import scenes

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("kind,n", [("plain", 100), ("plain", 3000), ("multi", 60)])
def test_old_dt_set_after_an_export(kind, n):
    sc = (scenes.plain_large_scene(n=n, seed=4) if kind == "plain" else
          scenes.multi_collider_scene(n=n, n_springs=5, n_joints=5, seed=4))
    out = []
    for export in (True, False):
        p, handles = sc.build_physics()
        p.step(sc.dt, 2)
        if export:
            p.bodies()
        else:
            p.get_rbd(int(handles[0]))
        p.old_dt = 0.004
        assert p.old_dt == np.float32(0.004)
        p.bodies()
        assert p.old_dt == np.float32(0.004)
        r = p.get_rbd(int(handles[1]))
        r.set_velocity((1.0, 2.0))
        p.set_rbd(int(handles[1]), r)  # the next step goes up from the mirror
        assert p.old_dt == np.float32(0.004)
        p.step(sc.dt, 2)
        out.append(p.bodies())
    for k in ("position", "position_old", "velocity", "rotation"):
        assert np.array_equal(bits(out[0][k]), bits(out[1][k])), k
