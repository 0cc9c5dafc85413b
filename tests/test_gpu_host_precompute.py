"""precompute_at() and the host's probe search need no device: in a process that has not
rendered yet they start none (a rank that picks its GPU afterwards, a parent that forks
its workers), and they give the tables that a running device makes."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_VIEWS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "views.json")))

CHILD = """
import json, os, sys
sys.path.insert(0, %r)
import newman_amd as nm
v = json.loads(%r)
def in_use():
    return any(os.path.realpath("/proc/self/fd/" + f) == "/dev/kfd" for f in os.listdir("/proc/self/fd"))
was = in_use()
m = nm.Mandelbrot(24, 32)
m.set_view(2900, v["re"], v["im"], "1e-16")
m.precompute_at(v["re"], v["im"])
h = nm.Mandelbrot(24, 32)
h.set_view(2900, v["re"], v["im"], "1e-16")
h.set_probe_mode(nm.PROBE_HOST)
h.precompute()
print("device", was, in_use())
m.computeAll()
print("after a render", in_use())
"""


def test_no_device_is_started(gpu):
    v = _VIEWS["t11"]
    code = CHILD % (ROOT, json.dumps({"re": v["re"], "im": v["im"]}))
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    was, now = out.stdout.splitlines()[0].split()[1:]
    assert out.stdout.splitlines()[1] == "after a render True"
    assert now == was == "False"


def test_the_tables_are_the_same(gpu):
    """The device's tables in this process against a host-only orbit's first entries."""
    v = _VIEWS["t11"]
    both = []
    for N in (2900, 1000):  # 1000: the host's work
        m = gpu.Mandelbrot(24, 32)
        m.set_view(N, v["re"], v["im"], "1e-16")
        m.precompute_at(v["re"], v["im"])
        both.append(m.reference())
    for long, short in zip(*both):
        assert np.array_equal(long[:len(short)], short)
