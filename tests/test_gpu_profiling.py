"""Stage times are those of the path a world steps on without them, and change no
result.
"""
import time

import numpy as np
import pytest

from blobs_amd import scenes
from blobs_amd.physics import Physics

pytestmark = pytest.mark.gpu
SUBSTEP, REBUILD = 0, 1


@pytest.mark.parametrize("n", [200, 1500, 5000])
@pytest.mark.parametrize("batch", [False, True])
def test_stage_times(n, batch):
    sc = scenes.plain_large_scene(n=n, seed=6)
    a, b = (Physics.batch([sc.build_physics()[0] for _ in range(3)]) if batch else sc.build_physics()[0]
            for _ in range(2))
    a.set_profiling(True)
    t = time.perf_counter()
    a.step(sc.dt, 3)
    if batch:
        a.step(sc.dt, 4)
    else:
        a.run_chunks(sc.dt, 4, 1)
    a.synchronize()
    wall = 1e3 * (time.perf_counter() - t)
    b.step(sc.dt, 7)
    (n_sub, ms_sub), (n_reb, ms_reb) = a.stage_stats(SUBSTEP), a.stage_stats(REBUILD)
    assert n_sub >= 3 * 8 and 0.0 < ms_sub + ms_reb < wall
    if n <= 2048:  # one workgroup a world: no grid, and so no rebuild of one
        assert n_sub == 7 * 8 and n_reb == 0
    else:
        assert n_reb > 0
    a.set_profiling(False)
    a.step(sc.dt, 1)
    b.step(sc.dt, 1)
    x, y = a.bodies(), b.bodies()
    for k in ("position", "velocity"):
        assert np.array_equal(x[k], y[k])
