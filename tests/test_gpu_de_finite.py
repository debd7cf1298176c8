"""Density estimation of 32-bit histograms whose values are not finite as floats."""
import ctypes

import numpy as np
import pytest

from test_gpu_de_taps import BANKS, _bank, _hist

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k1,k2", [(1068.0, -1.0 / 20000.0), (1e39, 1.0 / 2000.0)])
def test_float_values_that_are_not_finite(prod, k1, k2):
    """The brightest cells take the logarithm of a negative number, or pass the
    largest float: the exact mode's result, to the bit (a clamped tap would
    multiply them by zero)."""
    widths, coefs = _bank(BANKS["flame"])
    W, H = 90, 70
    b = _hist(np.random.default_rng(4), W, H, 33, 0.03)
    out = []
    for f in (prod.lib().fl3h_density_estimate, prod.lib().fl3h_density_estimate_production):
        acc = np.zeros((H, W, 4), dtype=np.float32)
        assert f(b.ctypes.data_as(ctypes.c_void_p), W, H, 33, 1, k1, k2, 0.4, len(widths) - 1, len(widths) - 1,
                 coefs.shape[1], len(widths), widths.ctypes.data_as(ctypes.c_void_p),
                 coefs.ctypes.data_as(ctypes.c_void_p), acc.ctypes.data_as(ctypes.c_void_p)) == 0, prod.last_error()
        out.append(acc)
    assert np.array_equal(out[0], out[1], equal_nan=True)
    assert not np.isfinite(out[1]).all() and np.isfinite(out[1]).any()
