"""Where a result above 1 MB goes: pinned host memory and device memory take the runtime's
own copy, ordinary memory at any alignment the pinned ring; every one gets the same bytes
and nothing around them is touched.  The comparison values come by copies of at most 1 MB,
which never take the ring."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

VIEW = (60, "-0.75", "0.1")


def _into(nm, m, widths, out_ptr):
    torch.cuda.synchronize()  # torch's own work on the destination is over
    arr = (C.c_char_p * len(widths))(*[w.encode() for w in widths])
    st = nm.RenderStats()
    assert nm.lib().nm_render_frames(m._h, arr, len(widths), 0, 0, 1, out_ptr, C.byref(st)) == 0


def _widths(n):
    return ["%.6f" % (3.0 / 1.1 ** k) for k in range(n)]


def _wanted(nm, nr, nc, widths):
    """Each frame's 8-byte entries (counts and smoothing bits): the device's own result,
    copied in slices of at most 1 MB by another library."""
    m = nm.Mandelbrot(nr, nc)
    m.set_view(*VIEW, "3.0")
    pinned = torch.empty(len(widths) * nr * nc, dtype=torch.int64, pin_memory=True)
    small = []
    for w in widths:
        one = torch.empty(nr * nc, dtype=torch.int64, device="cuda")
        _into(nm, m, [w], one.data_ptr())
        small += [one[k:k + 131072].cpu().numpy() for k in range(0, nr * nc, 131072)]
    _into(nm, m, widths, pinned.data_ptr())
    want = np.concatenate(small)
    assert np.array_equal(pinned.numpy(), want)
    return m, want


@pytest.mark.parametrize("nr,nc,frames", [(200, 300, 1),        # 0.5 MB: the runtime's copy
                                          (300, 701, 1),        # 1.7 MB
                                          (512, 2049, 1),       # 8.4 MB
                                          (600, 801, 6),        # 23.1 MB: 1 MB chunks
                                          (1000, 1111, 5)])     # 44 MB: 2 MB chunks, slots used again
def test_every_destination_gets_the_same_bytes(gpu, nr, nc, frames):
    widths = _widths(frames)
    m, want = _wanted(gpu, nr, nc, widths)
    size = 8 * nr * nc * frames
    for shift in (0, 4, 4096 + 12):  # the entries' own alignment is 4 bytes
        room = np.full(size + 8192 + 64, 0xA5, dtype=np.uint8)
        start = (-room.ctypes.data) % 4096 + shift
        _into(gpu, m, widths, room.ctypes.data + start)
        assert np.array_equal(room[start:start + size], want.view(np.uint8))
        assert np.all(room[:start] == 0xA5) and np.all(room[start + size:] == 0xA5)
    on_device = torch.full((nr * nc * frames + 2,), -1, dtype=torch.int64, device="cuda")
    _into(gpu, m, widths, on_device.data_ptr() + 8)
    got = on_device.cpu().numpy()
    assert np.array_equal(got[1:-1], want) and got[0] == -1 and got[-1] == -1


def test_images_into_pinned_memory(gpu):
    """colour() into memory of either kind: the same bytes."""
    m = gpu.Mandelbrot(900, 1300)
    m.set_view(*VIEW, "3.0")
    m.computeAll()
    pal = np.arange(180, dtype=np.uint8)
    want, _ = m.colour(pal.reshape(60, 3), smooth=True, sc=1)
    pinned = torch.zeros(900 * 1300 * 3, dtype=torch.uint8, pin_memory=True)
    assert gpu.lib().nm_colour(m._h, -1, pal.ctypes.data, 60, 1, 1, pinned.data_ptr(), None) == 0
    assert np.array_equal(pinned.numpy(), np.asarray(want).ravel())
