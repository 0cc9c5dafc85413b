"""The device's reference tables where the other order of operations shows: points at
which a coefficient cancels down to its last bits keep the chain's doubles, and all
tables of long orbits, remainders and floatexp forms among them, equal the oracle's."""
import json
import os

import numpy as np
import pytest

import oracle_lib as O
from test_orbit_bound import CRITICAL, critical_point

pytestmark = pytest.mark.gpu

_VIEWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))


def _pair(nm, N, width, re, im):
    m = nm.Mandelbrot(24, 32)
    m.set_view(N, re, im, width)
    m.precompute_at(re, im)
    o = O.OView(24, 32)
    o.set_view(N, re, im, width)
    o.precompute_at(re, im)
    n = m.reference_length()
    assert n == o.ref_len() and n >= 1024
    return m, o, n


def _short_remainders(nm, width, v):
    m = nm.Mandelbrot(24, 32)
    m.set_view(1000, v["re"], v["im"], width)
    m.precompute_at(v["re"], v["im"])
    return m.reference_tables()[0]


@pytest.mark.parametrize("k,lo,hi,beside", CRITICAL)
def test_a_cancelling_coefficient_is_the_chains(gpu, k, lo, hi, beside):
    c = critical_point(k, lo, hi, beside)
    m, o, _ = _pair(gpu, 1500, "1e-25", c, "0")
    for got, want in zip(m.reference()[1:], o.series()[2:]):
        assert np.array_equal(got, want), np.argwhere(got != want)[:4].ravel()


@pytest.mark.parametrize("name,width,N", [("t11", "1e-16", 2900), ("t13", "1e-25", 7900), ("c5_detail1", "1e-100", 50000),
                                          ("c3_detail1", "1e-200", 2000)])
def test_every_table_equals_the_oracles(gpu, name, width, N):
    v = _VIEWS[name]
    m, o, n = _pair(gpu, N, width, v["re"], v["im"])
    for got, want in zip(m.reference(), o.series()[1:]):
        assert np.array_equal(got, want[:2 * n])
    xlo, fx = m.reference_tables()
    for (gm, ge), (wm, we) in zip(fx, o.series_fx()):
        zero = wm == 0.0
        assert np.array_equal(gm, wm) and np.array_equal(ge[~zero], we[~zero])
    # what the nearest doubles leave of the orbit: at most half of their last bit, and
    # the host's values on the orbit's start (an orbit short enough to be its work)
    X = m.reference()[0]
    assert np.all(np.abs(xlo) <= np.spacing(np.abs(X)) / 2)
    short = _short_remainders(gpu, width, v)
    assert np.array_equal(xlo[:len(short)], short)
    m.set_series_mode(1)  # the floatexp tables in use
    assert m.reference_length() == n
