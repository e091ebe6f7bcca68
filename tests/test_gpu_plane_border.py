"""GPU: the interpolated planes and their 76-pixel border come from one launch
whose workgroups each make a tile of the core, a piece of the bands above and
below or of the strips at the sides.  Every plane's bytes, inside and outside
the padded picture, against the oracle:

* plane origins at every kind of position in a 64-byte line (the tiles start at
  such lines), widths and heights around one tile, one band piece and one strip
  piece;
* all planes, and the half-pel ones alone (the others are not touched);
* bytes outside the padded picture keep their values.
"""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from xavs2_amd import lib as X

pytestmark = pytest.mark.gpu

PAD = X.XME_PAD
GUARD = 0x5A


@pytest.mark.parametrize("w,h,shift,frac", [(8, 8, 0, 2), (56, 12, 4, 2), (64, 16, 16, 2), (72, 17, 20, 1),
                                            (48, 9, 60, 2), (136, 31, 36, 2), (200, 104, 44, 1), (264, 33, 12, 2)])
def test_planes_and_border_match_oracle(w, h, shift, frac):
    rng = np.random.default_rng(w * 1000 + h + shift)
    img = rng.integers(0, 256, (h, w), dtype=np.uint8)
    src = O.Plane(w, h)
    src.set_picture(img)
    src.expand_border()
    exp = O.interp_planes(src, frac)
    stride, rows = w + 2 * PAD + 68, h + 2 * PAD
    built = [k for k in range(1, 16) if frac == 2 or k in (2, 8, 10)]
    # the padded pictures start `shift` bytes into row 1 of their buffers
    buf = np.full((16, (rows + 2) * stride), GUARD, np.uint8)
    want = buf.copy()
    for k in [0] + built:
        for a in (buf, want) if k == 0 else (want,):
            win = np.lib.stride_tricks.as_strided(a[k, stride + shift:], (rows, w + 2 * PAD), (stride, 1))
            win[:] = exp[k].view()[:rows, : w + 2 * PAD]
    dev = X.upload(buf.ravel())
    ptrs = (C.c_void_p * 16)(*[dev.ptr + k * buf.shape[1] + stride + shift + PAD * stride + PAD for k in range(16)])
    assert X.lib().xme_interpolate_frame(ptrs, stride, w, h, frac, None) == X.XME_OK
    got = dev.download(buf.size, np.uint8).reshape(buf.shape)
    for k in range(16):
        assert np.array_equal(got[k], want[k]), k
