"""A render that is refused leaves the device's last result alone: the frames of another
object's last render are coloured as before, however large the refused set was."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAL = np.arange(192, dtype=np.uint8).reshape(64, 3)
DEEP = dict(re="0.13043143648640199241858146874999999999999999999999999999999999999999999999999999999999999999999900975e0",
            im="-0.5878286807333514631686996874999999999999999999999999999999999999999999999999999999999999999999941956e0")


def _small(nm, deep):
    m = nm.Mandelbrot(40, 60)
    if deep:
        m.set_view(64, DEEP["re"], DEEP["im"], "1e-25")
        m.precompute()
        widths = ["1e-25", "3e-25"]
    else:
        m.set_view(64, "-0.75", "0", "3")
        widths = ["3", "2"]
    m.render_frames(widths, copy_back=False)
    return m, [m.colour(PAL, smooth=True, sc=1, frame=k)[0] for k in range(2)]


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("deep", [False, True])
@pytest.mark.parametrize("fp32x", [False, True])
def test_the_last_result_outlives_a_refused_render(gpu, tile, deep, fp32x):
    nm = gpu
    big = nm.Mandelbrot(1500, 2000)
    if deep:
        big.set_view(64, DEEP["re"], DEEP["im"], "1e-25")
        big.precompute()
    else:
        big.set_view(64, "-0.75", "0", "3")
    if fp32x:
        big.set_delta_mode(nm.NM_DELTA_FP32X)
    big.set_launch(tile=tile)
    a, want = _small(nm, deep)
    # block sizes that no kernel has; a set that needs larger buffers than any before
    width = "1e-25" if deep else "3"
    for block in ((7, 64) if fp32x and deep else (7, 48)):
        with pytest.raises(nm.NewmanError):
            big.render_frames([width] * 3, block_k=block, copy_back=False)
        for k in range(2):
            assert np.array_equal(a.colour(PAL, smooth=True, sc=1, frame=k)[0], want[k])
    # a render that is done takes its place
    big.render_frames([width], copy_back=False)
    with pytest.raises(nm.NewmanError):
        a.colour(PAL, smooth=True, sc=1, frame=0)
