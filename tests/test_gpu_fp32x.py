"""FP32X deltas (FP32 mantissa pair + int32 exponent) on the GPU.

Bit-exact against the oracle's restatement of the same arithmetic; against the
FP64-delta kernel and the reference method, the per-sample count and smoothing
error is measured and bounded: FP32 carries 24 bits where FP64 carries 53, so
samples whose escape is decided by the last bits of a long chaotic orbit can
move.  The views include deltas far below the FP32 range (width 1e-40).
"""
import json
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

_VIEWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))
CASES = [("t13", 48, 64, "1e-25"), ("t13", 48, 64, "3e-23"), ("t11", 48, 64, "1e-15"), ("c4_seed1", 36, 48, "1e-40")]
# measured agreement of FP32X counts with the FP64 kernel, less a margin: the
# error grows with the length of the orbit after a sample leaves the reference
# (N 3000 for t11, 8000 for t13, 60000 for c4_seed1)
MIN_AGREE = {"t13": 0.999, "t11": 0.995, "c4_seed1": 0.97}
# the same for smoothing within 1e-3 where the counts agree
MIN_SMOOTH = {"t13": 0.98, "t11": 0.97, "c4_seed1": 0.90}


def _pair(name, nr, nc, width):
    import newman_amd as nm
    v = _VIEWS[name]
    m = nm.Mandelbrot(nr, nc)
    m.set_view(v["N"], v["re"], v["im"], width)
    m.precompute()
    o = O.OView(nr, nc)
    o.set_view(v["N"], v["re"], v["im"], width)
    o.precompute()
    return m, o


@pytest.mark.parametrize("name,nr,nc,width", CASES)
@pytest.mark.parametrize("K", [8, 12, 16])
def test_fp32x_bit_exact_vs_oracle(gpu, name, nr, nc, width, K):
    m, o = _pair(name, nr, nc, width)
    m.set_delta_mode(1)
    st = m.render(block_k=K)
    g = m.grid()
    rc = np.array([(r, c) for r in range(nr) for c in range(nc)], dtype=np.int32)
    ref = o.pert_samples_fx(rc, K).reshape(nr, nc)
    bad = np.argwhere(g["iterations"] != ref["iterations"])
    assert len(bad) == 0, (len(bad), bad[:5])
    assert np.array_equal(g["smoothing"].view(np.uint32), ref["smoothing"].view(np.uint32))
    assert st["block_k"] == K


def test_fp32x_refuses_64_step_blocks(gpu):
    """FP32X mantissas are renormalised at block ends: 64-step blocks are FP64 only."""
    nm = gpu
    m, _ = _pair(*CASES[0])
    m.set_delta_mode(1)
    with pytest.raises(nm.NewmanError) as e:
        m.render(block_k=64)
    assert e.value.code == nm.NM_ERR_ARG
    m.set_delta_mode(0)
    assert m.render(block_k=64)["block_k"] == 64


@pytest.mark.parametrize("name,nr,nc,width", CASES)
def test_fp32x_error_against_fp64_and_reference(gpu, name, nr, nc, width):
    """The per-sample error of FP32X deltas, reported and bounded: counts equal to
    the FP64-delta kernel and to the reference method (SA + HP continuation) on
    at least MIN_AGREE of the samples; where counts agree the smoothing differs by
    < 1e-3 on at least MIN_SMOOTH of them (long orbits after the reference shift
    the escape radius more than the count)."""
    m, o = _pair(name, nr, nc, width)
    m.render()
    g64 = m.grid().copy()
    m.set_delta_mode(1)
    m.render()
    g32 = m.grid().copy()
    ref = o.render_rows(np.arange(nr))
    same64 = g32["iterations"] == g64["iterations"]
    sameref = g32["iterations"] == ref["iterations"]
    ds = np.abs(g32["smoothing"].astype(np.float64) - g64["smoothing"])[same64]
    print("FP32X %s %s: counts = FP64 on %.4f%%, = reference on %.4f%%; max |count diff| %d; "
          "smoothing |diff| median %.2e p99 %.2e" % (
              name, width, 100 * same64.mean(), 100 * sameref.mean(),
              np.abs(g32["iterations"].astype(np.int64) - g64["iterations"]).max(),
              np.median(ds) if ds.size else 0.0, np.percentile(ds, 99) if ds.size else 0.0))
    bar = MIN_AGREE[name]
    assert same64.mean() >= bar
    assert sameref.mean() >= bar
    assert (ds < 1e-3).mean() >= MIN_SMOOTH[name]


def test_no_series_deltas_at_width_1e200(gpu):
    """Width 1e-200 (deltas ~1e-201, far below the FP32 range), N 50000: the
    reference's double-precision series test degenerates there (every index is
    stable, the whole frame skips to N), so both delta forms run the plain
    perturbation from d_0 = e (no series), 50000 steps per sample.  Each is
    bit-exact against the oracle; FP32X counts equal FP64 on >= 95% of samples
    (the measured error is printed).  The seeded walk's frame is uniform at this
    depth (every sample escapes with the reference, at 49999)."""
    import newman_amd as nm
    nr, nc, K = 24, 32, 8
    m, o = _pair("c3_seed1", nr, nc, _VIEWS["c3_seed1"]["width"])
    m.set_skip_mode(nm.SKIP_NONE, 16)
    rc = np.array([(r, c) for r in range(nr) for c in range(nc)], dtype=np.int32)
    ua = np.ones(len(rc), dtype=np.int32)
    m.render(block_k=K)
    g64 = m.grid().copy()
    ref64 = o.pert_samples_ua(rc, ua).reshape(nr, nc)
    assert np.array_equal(g64["iterations"], ref64["iterations"])
    assert np.array_equal(g64["smoothing"].view(np.uint32), ref64["smoothing"].view(np.uint32))
    m.set_delta_mode(1)
    m.render(block_k=K)
    g32 = m.grid().copy()
    ref32 = o.pert_samples_fx(rc, K, ua).reshape(nr, nc)
    assert np.array_equal(g32["iterations"], ref32["iterations"])
    assert np.array_equal(g32["smoothing"].view(np.uint32), ref32["smoothing"].view(np.uint32))
    same = g32["iterations"] == g64["iterations"]
    print("FP32X vs FP64 at 1e-200 (no series): counts equal on %.3f%%, max |diff| %d" % (
        100 * same.mean(), np.abs(g32["iterations"].astype(np.int64) - g64["iterations"]).max()))
    assert same.mean() >= 0.95


@pytest.mark.parametrize("K", [8, 12, 16, 32])
@pytest.mark.parametrize("name,nr,nc,width,N", [("t13", 31, 70, "3e-23", 8000), ("t13", 31, 70, "1e-24", 7990),
                                                ("t11", 33, 65, "1e-15", 3000)])
def test_blocks_between_refills_keep_results(gpu, name, nr, nc, width, N, K):
    """Up to 64 steps of blocks run between refills where the series is in floatexp, up
    to 32 where it is in doubles, past an escape, the orbit's end and the limit N (also
    where it falls inside them): grids and step counts of the oracle's single blocks."""
    import newman_amd as nm
    v = _VIEWS[name]
    m, o = nm.Mandelbrot(nr, nc), O.OView(nr, nc)
    for x in (m, o):
        x.set_view(N, v["re"], v["im"], width)
    m.precompute()
    o.precompute_at(*m.reference_point())
    m.set_delta_mode(1)
    rc = np.array([(r, c) for r in range(nr) for c in range(nc)], dtype=np.int32)
    want = o.pert_samples_fx(rc, K).reshape(nr, nc)
    stats = []
    for mode in (nm.NM_SERIES_DOUBLE, nm.NM_SERIES_FLOATEXP):
        m.set_series_mode(mode)
        stats.append(m.render(block_k=K))
        g = m.grid()
        assert np.array_equal(g["iterations"], want["iterations"])
        assert np.array_equal(g["smoothing"].view(np.uint32), want["smoothing"].view(np.uint32))
    for k in ("executed", "credited", "n_rebased"):
        assert stats[0][k] == stats[1][k], k
