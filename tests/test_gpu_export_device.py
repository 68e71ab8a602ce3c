"""A bulk read of a world whose device is not the caller's current one."""
import threading

import numpy as np
import pytest

from blobs_amd import scenes

torch = pytest.importorskip("torch")
pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two devices")]


@pytest.mark.parametrize("n", [100, 60000])
def test_read_from_another_device(n):
    sc = scenes.plain_large_scene(n=n, seed=4)
    torch.cuda.set_device(1)
    try:
        a, b = sc.build_physics()[0], sc.build_physics()[0]
        for w in (a, b):
            w.step(sc.dt, 2)
        here = a.bodies()
        torch.cuda.set_device(0)
        there = b.bodies()
        assert torch.cuda.current_device() == 0
        out = []
        thread = threading.Thread(target=lambda: out.append(b.bodies()))  # (its current device is the first)
        thread.start()
        thread.join()
        for k in ("position", "velocity"):
            assert np.array_equal(here[k], there[k]) and np.array_equal(here[k], out[0][k])
    finally:
        torch.cuda.set_device(0)
