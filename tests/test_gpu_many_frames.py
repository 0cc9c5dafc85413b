"""Frame sets of more frames than the staging buffer takes at a time: every frame equals
its own render, and what the engine keeps for a set of many small frames stays small."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

RE = "0.13043143648640199241858146874999999999999999999999999999999999999999999999999999999999999999999900975e0"
IM = "-0.5878286807333514631686996874999999999999999999999999999999999999999999999999999999999999999999941956e0"
BATCH = 4096


@pytest.mark.parametrize("deep", [False, True])
@pytest.mark.parametrize("frames", [BATCH - 1, BATCH, BATCH + 1, 2 * BATCH + 3])
def test_frames_at_the_batches_edges(gpu, frames, deep):
    m = gpu.Mandelbrot(3, 5)
    if deep:
        m.set_view(3000, RE, IM, "1e-25")
        m.precompute()
        widths = ["%.9fe-25" % (1.0 + k / 1000.0) for k in range(frames)]
    else:
        m.set_view(200, "-0.75", "0.05", "3")
        widths = ["%.9f" % (3.0 / (1.0 + k / 1000.0)) for k in range(frames)]
    got, _ = m.render_frames(widths)
    edges = sorted({0, 1, BATCH - 2, BATCH - 1, BATCH, BATCH + 1, 2 * BATCH - 1, 2 * BATCH, frames - 1})
    for k in [k for k in edges if k < frames]:
        one, _ = m.render_frames([widths[k]])
        assert np.array_equal(one[0], got[k]), k


def test_many_small_frames_keep_little_memory(gpu):
    m = gpu.Mandelbrot(1, 2)
    m.set_view(50, "-0.75", "0.05", "3")
    widths = ["%.9f" % (3.0 / (1.0 + k / 1000.0)) for k in range(40000)]
    m.render_frames(widths[:2])
    before = torch.cuda.mem_get_info()[0]
    m.render_frames(widths, copy_back=False)
    # 2 KB a frame would be 81 MB; the records, tables and states take some 20
    assert before - torch.cuda.mem_get_info()[0] < 48 << 20
