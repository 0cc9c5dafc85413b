"""Persistent waves per SIMD on the series path: a CU holds 4, whatever is asked for; the
statistics and the autotuner's rows give what ran, and the grids do not depend on it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RE = "0.13043143648640199241858146874999999999999999999999999999999999999999999999999999999999999999999900975e0"
IM = "-0.5878286807333514631686996874999999999999999999999999999999999999999999999999999999999999999999941956e0"


@pytest.mark.parametrize("mode", [0, 1])
def test_the_series_path_runs_what_it_reports(gpu, mode):
    m = gpu.Mandelbrot(150, 200)
    m.set_view(8000, RE, IM, "1e-25")
    m.set_delta_mode(mode)
    m.precompute()
    m.computeAll()
    want = m.grid().copy()
    for asked in (1, 2, 3, 4, 5, 8, 16):
        st = m.render(waves_per_simd=asked)
        assert st["waves_per_simd"] == min(asked, 4)
        assert np.array_equal(m.grid(), want)
    m.set_launch(waves_per_simd=8)
    assert m.render()["waves_per_simd"] == 4 and np.array_equal(m.grid(), want)


def test_the_autotuner_sweeps_what_runs(gpu):
    m = gpu.Mandelbrot(60, 80)
    m.set_view(2000, RE, IM, "1e-25")
    m.precompute()
    best, table = m.autotune_frames(["1e-25", "4e-25"])
    assert {r["waves_per_simd"] for r in table} == {1, 2, 3, 4}
    assert m.render()["waves_per_simd"] == best["waves_per_simd"]
