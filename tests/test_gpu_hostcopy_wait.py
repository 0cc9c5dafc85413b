"""A render that takes long and returns many MB: its result's helper threads sleep
until the first bytes are there, so that the call holds one core, not four."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_helpers_sleep_while_the_render_runs(gpu):
    m = gpu.Mandelbrot(1920, 2720)  # 42 MB: more than the ring
    # inside the period-3 bulb: every sample runs all N updates (5.2e6 x 7e5, some 0.6 s)
    m.set_view(700000, "-0.1225611668766536", "0.7448617666197442", "0.01")
    m.N = 100
    m.computeAll()  # the ring and its threads are there
    m.N = 700000
    cpu, wall = time.process_time(), time.perf_counter()
    m.computeAll()
    cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    assert np.all(m.grid()["iterations"] == 700000)
    # the caller's wait, and half as much again for the runtime's own threads
    assert cpu < 1.5 * wall, (cpu, wall)
