"""Large results reach the caller through a pinned ring that several threads empty:
sizes around its threshold (1 MB), its pieces (256 KB), its chunks (1 and 2 MB) and its
32 MB, each against the same frames rendered one at a time into small copies."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nc,frames", [(256, 512, 1),       # 1 MB: the last size of the runtime's copy
                                          (1, 131073, 1),      # 8 bytes past it: a chunk and a piece of 8 bytes
                                          (300, 701, 1),       # 1.7 MB: a ragged last piece
                                          (512, 2048, 1),      # 8 MB: whole chunks
                                          (512, 2049, 1),      # and a little more
                                          (600, 801, 6),       # 23.1 MB: 1 MB chunks, a ragged last one
                                          (1024, 1023, 4),     # 32.7 MB in 2 MB chunks: most of the ring
                                          (1000, 1111, 9)])    # 80 MB: the ring's slots are used again
def test_large_results(gpu, nr, nc, frames):
    m = gpu.Mandelbrot(nr, nc)
    m.set_view(60, "-0.75", "0.1", "3.0")
    widths = ["%.6f" % (3.0 / 1.1 ** k) for k in range(frames)]
    for _ in range(2):  # the second time the ring and its threads are there
        got, _ = m.render_frames(widths)
        one = gpu.Mandelbrot(nr, nc)
        for k, w in enumerate(widths):
            one.set_view(60, "-0.75", "0.1", w)
            one.render(copy_back=False)
            # the escape counts of a frame as bytes of its image: 3 bytes a sample
            pal = np.arange(180, dtype=np.uint8).reshape(60, 3)
            img, _ = one.colour(pal, smooth=False, sc=1)
            want = np.vstack([pal, np.zeros((1, 3), np.uint8)])[got[k]["iterations"]]
            assert np.array_equal(img, want)
