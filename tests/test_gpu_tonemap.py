"""The tone map's tiles in LDS against its direct reads, at the edges of a tile
(32 x 4 pixels)."""
import ctypes

import numpy as np
import pytest

from flam3_amd._lib import fl3h_tonemap_params

pytestmark = pytest.mark.gpu

PAD = 64     # taps across from which a tile's cells pass the LDS space


def _tonemap(prod, acc, bits, iw, ih, ss, off, filt, bpc):
    H, W, _ = acc.shape
    tp = fl3h_tonemap_params(image_width=iw, image_height=ih, oversample=ss, de_offset=off,
                             filter_width=filt.shape[0], nchan=4, transp=1, bytes_per_channel=bpc, earlyclip=0,
                             g=0.25, linrange=0.01, vibrancy=0.7, highpow=1.0)
    out = np.zeros((ih, iw, 4), dtype=np.uint16 if bpc == 2 else np.uint8)
    a, f = acc.copy(), np.ascontiguousarray(filt).ravel()
    vp = ctypes.c_void_p
    assert prod.lib().fl3h_tonemap(a.ctypes.data_as(vp), W, H, bits, ctypes.byref(tp), f.ctypes.data_as(vp),
                                   out.ctypes.data_as(vp)) == 0, prod.last_error()
    return out


@pytest.mark.parametrize("bits", [33, 64])
@pytest.mark.parametrize("iw,ih,ss,fw,off", [
    (1, 1, 1, 1, 0), (31, 3, 2, 4, 3), (32, 4, 3, 5, 1), (33, 5, 3, 5, 0), (70, 9, 4, 9, 2), (65, 4, 1, 3, 5),
    (32, 13, 5, 3, 0)])
def test_tiles_against_direct_reads(prod, bits, iw, ih, ss, fw, off):
    """Weights of zero beyond the filter add nothing to a sum and send the call
    to the kernel that reads every tap from memory: the same bytes."""
    rng = np.random.default_rng(iw * 100 + ih)
    W, H = off + (iw - 1) * ss + PAD + 1, off + (ih - 1) * ss + PAD
    acc = (rng.uniform(0, 1, (H, W, 4)) ** 4 * 300).astype(np.float32 if bits == 33 else np.float64)
    filt = rng.uniform(0.1, 1, (fw, fw))
    filt /= filt.sum()
    wide = np.zeros((PAD, PAD))
    wide[:fw, :fw] = filt
    for bpc in (1, 2):
        got = _tonemap(prod, acc, bits, iw, ih, ss, off, filt, bpc)
        want = _tonemap(prod, acc, bits, iw, ih, ss, off, wide, bpc)
        assert got.any()
        np.testing.assert_array_equal(got, want)
