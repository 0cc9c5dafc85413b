"""The reference tables' passes (chunks on three levels) on the host, against the chain
of high-precision operations that they stand for: every value lies within the bound
that decides whether the device's doubles are kept, tables that it keeps have equal
entries, and where a coefficient cancels down to its last bits it keeps none."""
import ctypes as C
import json
import os
from fractions import Fraction

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "newman_amd", "libnm_index_check.so")
_VIEWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))


def _check(re, im, limbs, n, cancel=0):
    if not os.path.exists(LIB):
        from newman_amd import build
        build.build_index_check()
    f = C.CDLL(LIB).nm_orbit_check
    f.restype = C.c_longlong
    f.argtypes = [C.c_char_p, C.c_char_p, C.c_int, C.c_int, C.c_int, C.POINTER(C.c_longlong)]
    out = (C.c_longlong * 5)()
    assert f(re.encode(), im.encode(), limbs, n, cancel, out) == 0
    accepted, differ, cancelled, outside, _ = list(out)
    assert outside == 0
    assert not accepted or differ == 0
    return accepted, differ, cancelled


def critical_point(k, lo, hi, beside):
    """A real c with dz_k/dc = 0 between lo and hi, so that A_k cancels; beside > 0:
    2^-beside off it, which leaves A_k some of its bits.  To 110 digits."""
    P = 1200

    def a(c):
        x, v = c, 1 << P
        for _ in range(k):
            v = ((2 * x * v) >> P) + (1 << P)
            x = ((x * x) >> P) + c
        return v
    lo, hi = (int(v * 2 ** 60) << (P - 60) for v in (lo, hi))
    up = a(lo) > 0
    assert up != (a(hi) > 0)
    while hi - lo > 2:
        mid = (lo + hi) // 2
        if (a(mid) > 0) == up:
            lo = mid
        else:
            hi = mid
    c = Fraction(lo, 1 << P) + (Fraction(1, 1 << beside) if beside else 0)
    n = int(-c * 10 ** 110)
    return "-%d.%s" % (n // 10 ** 110, str(n % 10 ** 110).zfill(110))


# (k, an interval where A_k changes its sign, how far beside): at 4 limbs A_k loses all
# of its bits, or all but some 56 of them, whose last ones go by the order of operations
CRITICAL = [(14, -1.567641, -1.567640, 0), (16, -1.531735, -1.531734, 0), (14, -1.567641, -1.567640, 221),
            (16, -1.531735, -1.531734, 221), (45, -1.530969, -1.530968, 238), (45, -1.530969, -1.530968, 239),
            (45, -1.530969, -1.530968, 240)]


@pytest.mark.parametrize("name,limbs,n", [("t11", 3, 2900), ("t13", 4, 7900), ("t13", 4, 1024), ("t13", 4, 1332),
                                          ("c4_seed1", 5, 3000), ("c5_detail1", 8, 50000), ("c3_detail1", 13, 2000)])
def test_the_views_orbits_are_kept(name, limbs, n):
    v = _VIEWS[name]
    assert _check(v["re"], v["im"], limbs, n)[0]


@pytest.mark.parametrize("re,im", [("-1.75", "0"), ("-1.9", "0"), ("-0.125", "0.75"), ("0", "1"), ("-2", "0"),
                                   ("-0.5", "0"), ("0.3", "0.6")])
def test_exact_and_escaping_points(re, im):
    _check(re, im, 4, 1500)


@pytest.mark.parametrize("every", [7, 13, 50, 333])
@pytest.mark.parametrize("limbs", [4, 8, 16])
def test_steps_that_cancel_to_a_doubles_last_bits(limbs, every):
    v = _VIEWS["t13"]
    accepted, _, cancelled = _check(v["re"], v["im"], limbs, 2000, every)
    assert accepted and cancelled > 50


@pytest.mark.parametrize("k,lo,hi,beside", CRITICAL)
def test_a_coefficient_that_cancels_away(k, lo, hi, beside):
    accepted, differ, cancelled = _check(critical_point(k, lo, hi, beside), "0", 4, 1500)
    assert cancelled > 190 and not accepted and differ
