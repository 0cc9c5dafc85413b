"""A reference's tables made on the device (orbits of at least 1024 entries) against
the oracle's chain of high-precision operations: every double equal.

The device takes the recurrences in chunks on three levels, so the sizes are around
its shortest orbit and around cubes (where the chunk grows), the precisions those of
each number of limbs it is compiled for, and the points include ones whose orbits are
short exact numbers, where the coefficients hang on their last bits and the host makes
the tables."""
import json
import os

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

_VIEWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))


def _same(nm, N, width, re, im, long=True):
    m = nm.Mandelbrot(24, 32)
    m.set_view(N, re, im, width)
    m.precompute_at(re, im)
    o = O.OView(24, 32)
    o.set_view(N, re, im, width)
    o.precompute_at(re, im)
    n = m.reference_length()
    assert n == o.ref_len() and (n >= 1023 or not long)
    X, A, B, C = m.reference()
    _, Xn, OA, OB, OC = o.series()
    assert np.array_equal(X, Xn[:2 * n])
    for got, want in ((A, OA), (B, OB), (C, OC)):
        assert np.array_equal(got, want), np.argwhere(got != want)[:4].ravel()


@pytest.mark.parametrize("name,width,N", [
    ("t11", "1e-16", 2900),           # 3 limbs
    ("t13", "1e-25", 7900),           # 4
    ("t13", "1e-25", 1023), ("t13", "1e-25", 1024), ("t13", "1e-25", 1025), ("t13", "1e-25", 1026),
    ("t13", "1e-25", 1332), ("t13", "1e-25", 1333),   # 11^3 steps and one more
    ("c4_seed1", "1e-40", 3000),      # 5 of 6
    ("c5_detail1", "1e-80", 2000),    # 7 of 8
    ("c5_detail1", "1e-100", 2500),   # 8
    ("c5_detail1", "1e-110", 1500),   # 9 of 16
    ("c3_detail1", "1e-200", 2000),   # 13 of 16
    ("c3_detail1", "1e-270", 1500),   # 17: the host's
])
def test_tables_equal_the_oracles(gpu, name, width, N):
    v = _VIEWS[name]
    _same(gpu, N, width, v["re"], v["im"])


@pytest.mark.parametrize("re,im", [("-2", "0"), ("0", "1"), ("-1", "0"), ("0", "0"), ("0.25", "0"), ("-1.75", "0"),
                                   ("-1.5", "0"), ("-0.125", "0.75")])
def test_exact_points_equal_the_oracles(gpu, re, im):
    _same(gpu, 1500, "1e-25", re, im, long=False)
