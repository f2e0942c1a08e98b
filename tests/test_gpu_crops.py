"""The crops' recogniser inputs in one launch (`crop_rec_kernel`) against the
crop and then its input: tiles that end past the crop and past the tensor,
crops under, about and over twice the tensor's height, turned ones, and
windows that leave the page on each side. The same bytes throughout."""
import ctypes as C

import numpy as np
import pytest

from ppocr_native_amd import images
from ppocr_native_amd.devmem import DeviceArray, synchronize

pytestmark = pytest.mark.gpu


def quad(x, y, w, h, t):
    c, s = np.cos(t), np.sin(t)
    return [[x, y], [x + w * c, y + w * s], [x + w * c - h * s, y + w * s + h * c], [x - h * s, y + h * c]]


def test_crop_rec_tiles():
    rng = np.random.default_rng(4)
    page = rng.integers(0, 256, (700, 1500, 3), dtype=np.uint8)
    qs = [quad(30, 20, 7, 5, 0), quad(40, 60, 333, 24, 0.01), quad(60, 100, 401, 48, -0.02), quad(10, 200, 900, 97, 0.02),
          quad(100, 150, 1200, 150, 0), quad(20, 30, 1300, 420, 0.05), quad(300, 40, 40, 500, 0.01),
          quad(900, 20, 130, 600, 0), quad(-30, -20, 200, 40, 0.1), quad(1390, 660, 200, 60, 0.2), quad(0, 0, 1500, 700, 0)]
    for cap in (0, 320):
        flat = np.ascontiguousarray(np.asarray(qs, np.float32))
        sizes = [images.crop_size(q) for q in flat]
        widths = [images.rec_width_fit(w, h, cap)[0] for w, h in sizes]
        d = DeviceArray.of(page.reshape(-1))
        outs = [DeviceArray.of(np.full(48 * w * 3, 7, np.float32)) for w in widths]
        n = len(qs)
        rc = images._sig().ppocr_hip_crop_rec_inputs(
            d.addr, 1500, 700, flat.ctypes.data_as(C.POINTER(C.c_float)), n, cap, (C.c_void_p * n)(*[o.addr for o in outs]),
            (C.c_size_t * n)(*[48 * w * 3 for w in widths]), (C.c_size_t * n)(), None)
        assert rc == 0
        synchronize()
        for q, o, w in zip(flat, outs, widths):
            want = images.rec_input(images.crop_text(page, q), cap)
            assert np.array_equal(o.download(48 * w * 3).reshape(48, w, 3), want)
