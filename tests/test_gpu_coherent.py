"""The steps that a wave's samples do together in the series start kernel, bit for
bit against the oracle's per-sample iteration: iteration limits inside, at and just
past a block of them, frames with fewer lanes than take part and ragged waves, a
bailout that leaves no room for the proof, and a reference that escapes early."""
import json
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

_VIEWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))


def _check(gpu, nr, nc, N, width, bailout=None, view="t13", point=None, fx=False):
    v = _VIEWS[view]
    m, o = gpu.Mandelbrot(nr, nc), O.OView(nr, nc)
    for x in (m, o):
        x.set_view(N, v["re"], v["im"], width)
        if bailout:
            x.set_bailout(bailout)
        x.set_series_mode(1 if fx else 0)
    if point:
        m.precompute_at(*point)
    else:
        m.precompute()
    o.precompute_at(*m.reference_point())
    st = m.render()
    rc = np.array([(r, c) for r in range(nr) for c in range(nc)], dtype=np.int32)
    want = o.render_samples(rc, pert=True).reshape(nr, nc)
    g = m.grid()
    assert np.array_equal(g["iterations"], want["iterations"])
    a, b = g["smoothing"].astype(np.float64), want["smoothing"].astype(np.float64)
    assert (np.abs(a - b) <= 1e-6 * np.maximum(np.abs(b), 1.0)).all()
    return st


@pytest.mark.parametrize("N", [7886, 7890, 7895, 7896, 7897, 7898, 7904, 7920, 8000])
@pytest.mark.parametrize("fx", [False, True])
def test_iteration_limits(gpu, N, fx):
    _check(gpu, 9, 100, N, "1e-24", fx=fx)


@pytest.mark.parametrize("nr,nc", [(1, 35), (1, 36), (1, 64), (5, 67), (40, 48)])
def test_lanes(gpu, nr, nc):
    st = _check(gpu, nr, nc, 8000, "1e-24")
    if nr * nc < 36:  # the fewest lanes that go together
        assert st["executed_start"] == 0
    elif nr * nc > 1000:
        assert st["executed_start"] > 0


@pytest.mark.parametrize("bailout", [1.5, 2.0, 3.0, 1e6, 1e160])
def test_bailouts(gpu, bailout):
    _check(gpu, 9, 100, 8000, "1e-24", bailout=bailout)


def test_reference_that_escapes(gpu):
    """The frame's corner as the reference: samples meet the end of its orbit."""
    v = _VIEWS["t13"]
    m = gpu.Mandelbrot(16, 64)
    m.set_view(8000, v["re"], v["im"], "1e-23")
    m.precompute()
    m.render()
    r, c = np.unravel_index(np.argmin(m.grid()["iterations"]), (16, 64))
    _check(gpu, 16, 64, 8000, "1e-23", point=m.pointAt(int(r), int(c)))
