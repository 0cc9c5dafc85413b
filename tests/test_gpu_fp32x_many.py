"""FP32X deltas on many samples run on smaller workgroups with smaller orbit windows: a
frame set on either side of that line equals its frames rendered one at a time, bit for
bit, for every block size, series form and sample order, with the same counts of steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VIEWS = {
    "walk-25": (8000, "1e-25",
                "0.13043143648640199241858146874999999999999999999999999999999999999999999999999999999999999999999900975e0",
                "-0.5878286807333514631686996874999999999999999999999999999999999999999999999999999999999999999999941956e0"),
    # an orbit longer than both windows together
    "walk-30": (20000, "1e-30",
                "0.32774381527122875535040797894265624999999999999999999999999999999999999999999999999999999999999702733e0",
                "-0.5099534897928655695535697145158348437499999999999999999999999999999999999999999999999999999999933861e0"),
}


@pytest.mark.parametrize("view,block,series,tile,nr,nc,frames,many", [
    ("walk-25", 0, 0, 0, 1024, 1024, 4, True),      # 2^22 samples
    ("walk-25", 0, 0, 0, 2047, 2049, 1, False),     # one less
    ("walk-25", 8, 1, 0, 1001, 1051, 4, True),
    ("walk-25", 12, 0, 32, 1001, 1051, 4, True),
    ("walk-30", 16, 0, 0, 1001, 1051, 4, True),
    ("walk-30", 32, 1, 64, 1001, 1051, 4, True),
    ("walk-30", 0, 0, 0, 1001, 1051, 4, True),
])
def test_sets_equal_their_frames(gpu, view, block, series, tile, nr, nc, frames, many):
    N, width, re, im = VIEWS[view]
    m = gpu.Mandelbrot(nr, nc)
    m.set_view(N, re, im, width)
    m.set_delta_mode(gpu.NM_DELTA_FP32X)
    m.set_series_mode(series)
    m.precompute()
    m.set_launch(block_k=block, tile=tile)
    widths = ["%.2fe%s" % (1.0 + 0.8 * k, width[2:]) for k in range(frames)]
    whole, st = m.render_frames(widths)
    assert st["waves_per_simd"] == (6 if many else 4) and st["n_iterated"] > 0
    total = {k: 0 for k in ("executed", "credited", "skipped", "n_iterated", "n_rebased")}
    for k, w in enumerate(widths):
        one, s = m.render_frames([w]) if frames > 1 else m.render_frames([w], waves_per_simd=2)
        assert np.array_equal(one[0], whole[k])
        for key in total:
            total[key] += s[key]
    assert total == {k: st[k] for k in total}
