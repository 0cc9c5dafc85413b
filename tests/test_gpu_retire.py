"""Escaped samples leave the iterate kernels through a queue per wave that is
smoothed 64 at a time: list lengths around a wave and a queue, on both paths,
against the oracle.  At the plain view every sample outlives the start kernel."""
import json
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

_T13 = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))["t13"]


def _check(g, want):
    assert np.array_equal(g["iterations"], want["iterations"])
    a, b = g["smoothing"].astype(np.float64), want["smoothing"].astype(np.float64)
    assert (np.abs(a - b) <= 1e-6 * np.maximum(np.abs(b), 1.0)).all()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 127, 128, 129, 4097])
@pytest.mark.parametrize("deep", [False, True])
def test_queue_lengths(gpu, n, deep):
    m, o = gpu.Mandelbrot(1, n), O.OView(1, n)
    view = (_T13["N"], _T13["re"], _T13["im"], "1e-24") if deep else (900, "-0.7453", "0.1127", "0.01")
    m.set_view(*view)
    o.set_view(*view)
    if deep:
        m.precompute()
        o.precompute_at(*m.reference_point())
    st = m.render()
    rc = np.array([(0, c) for c in range(n)], dtype=np.int32)
    want = o.render_samples(rc, pert=True) if deep else o.render_rows(np.zeros(1, dtype=np.int32))[0]
    _check(m.grid()[0], want)
    # cardioid and bulb samples are counted apart from credited work
    assert st["credited"] == int(want["iterations"].astype(np.int64).sum()) - st["n_cardioid"] * view[0]


@pytest.mark.parametrize("nr,nc", [(1023, 1024), (1024, 1024), (1024, 1025), (4100, 4100)])
def test_scatter_around_the_scan(gpu, nr, nc):
    """Up to 1024 start tiles the scatter sums the counts before its tile itself;
    beyond, the scan does, in one group of 16384 counts or (16.8 M samples) two."""
    m, o = gpu.Mandelbrot(nr, nc), O.OView(nr, nc)
    view = (60, "-0.75", "0.1", "3.0")
    m.set_view(*view)
    o.set_view(*view)
    st = m.render()
    rows = np.arange(nr, dtype=np.int32)[::1 if nr < 2000 else 16]
    want = o.render_rows(rows)
    _check(m.grid()[rows], want)
    assert st["n_iterated"] + st["n_cardioid"] + st["n_sa_resolved"] == nr * nc


@pytest.mark.parametrize("k", [8, 16, 32, 64])
@pytest.mark.parametrize("bailout", [1.5, 3.0, 1024.0, 2.0 ** 30, 2.0 ** 31])
def test_groups_that_overflow(gpu, k, bailout):
    """A group of up to 16 updates tests its last one: past an escape the values
    square themselves to infinity and NaN within it, and a limit may fall inside it.
    Counts are those of a test after every update (which radii below 2 and above 2^30
    have here, too)."""
    for N in (77, 130, 901):
        m, o = gpu.Mandelbrot(30, 47), O.OView(30, 47)
        for v in (m, o):
            v.set_view(N, "-0.7453", "0.1127", "0.3")
            v.set_bailout(bailout)
        m.render(block_k=k)
        assert np.array_equal(m.grid()["iterations"], o.render_rows(np.arange(30, dtype=np.int32))["iterations"])


@pytest.mark.parametrize("nr,nc,count", [(1, 1, 1), (1, 65, 1), (7, 19, 3), (256, 512, 1), (257, 511, 1), (64, 64, 33)])
@pytest.mark.parametrize("bailout", [1.5, 1024.0])
def test_small_sets_in_one_launch(gpu, nr, nc, count, bailout):
    """Up to 131072 samples of the plain path take one launch, more the usual kernels;
    a launch setting always takes those: the same grids and the same counts, frames
    that share a wave among them, and the oracle's."""
    m, o = gpu.Mandelbrot(nr, nc), O.OView(nr, nc)
    widths = ["%.6f" % (3.0 / 1.3 ** k) for k in range(count)]
    for N in (13, 16, 300):
        for v in (m, o):
            v.set_view(N, "-0.6", "0.4", "3.0")
            v.set_bailout(bailout)
        got, st = m.render_frames(widths)
        want, usual = m.render_frames(widths, block_k=64)
        assert np.array_equal(got, want)
        for k in ("n_cardioid", "n_sa_resolved", "n_iterated", "executed", "executed_start", "credited", "n_rebased"):
            assert st[k] == usual[k], k
        assert np.array_equal(got[0]["iterations"], o.render_rows(np.arange(nr, dtype=np.int32))["iterations"])
