"""The production density estimation's tables and clamped taps against the
exact mode, which looks every tap up in the filter bank: at the edges of a
workgroup's region, with one and two cells per lane, and with the tables in
LDS and outside it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bank(widths, cut=0):
    """Kernel i falls off radially to widths[i]; its rows `cut` entries short
    of what its radius asks for."""
    half = int(np.ceil(max(widths))) - 1
    ks = max((half + 1) * (half + 2) // 2 - cut, 1)
    coefs = np.zeros((len(widths), ks))
    for i, w in enumerate(widths):
        n = 0
        for hi in range(half + 1):
            for lo in range(hi + 1):
                if n < ks:
                    coefs[i, n] = max(1.0 - np.hypot(hi, lo) / (w + 0.3), 0.0) / (w * w + 0.2)
                n += 1
    return np.array(widths, dtype=np.float64), coefs


BANKS = {
    "flame": [9.0 * (i + 1) ** -0.4 for i in range(40)],     # the usual kind: in LDS as floats and as doubles
    "wide": [27.0 * (i + 1) ** -0.2 for i in range(60)],     # outside it
    "points": [1.0, 0.9, 0.4],                               # a source reaches its own cell
    "one": [4.5, 4.5],
}


@pytest.mark.parametrize("bits", [33, 64])
@pytest.mark.parametrize("W,H,bank,fill", [
    (1, 1, "flame", 1.0), (7, 5, "flame", 1.0), (8, 16, "one", 0.5), (9, 17, "flame", 0.3),
    (16, 16, "points", 0.7), (33, 31, "wide", 1.0), (65, 130, "flame", 0.02), (257, 64, "flame", 1.0),
    (97, 40, "wide", 0.2), (1039, 1025, "flame", 0.1), (1025, 1039, "points", 0.5), (2049, 513, "wide", 0.01),
    (2049, 2033, "flame", 0.05)])
def test_taps_against_the_bank(prod, bits, W, H, bank, fill):
    """Both sum the same non-negative terms in the same order, so they differ
    by at most the roundings of each sum, one or three per term, and of the
    terms' factors."""
    _compare(prod, bits, W, H, _bank(BANKS[bank]), fill)


@pytest.mark.parametrize("bits", [33, 64])
def test_rows_shorter_than_their_radius(prod, bits):
    """A bank whose rows lack their radius' last entries: its taps go on in
    the next row.  (Its last row has no next one, and no source.)"""
    widths, coefs = _bank([3.0, 3.0, 3.0, 0.9], cut=2)
    _compare(prod, bits, 90, 40, (widths, coefs), 0.5, mfi=2)


@pytest.mark.parametrize("value", [np.inf, np.nan, -np.inf])
def test_sources_that_are_not_finite(prod, value):
    """Infinities and NaN in a double histogram: the exact mode's result, to
    the bit (a clamped tap would multiply them by zero)."""
    widths, coefs = _bank(BANKS["flame"])
    b = _hist(np.random.default_rng(3), 70, 50, 64, 0.4)
    b[20, 30, :] = 255.0
    b[20, 30, 1] = value
    exact, got = _both(prod, b, 64, widths, coefs)
    assert np.array_equal(exact, got, equal_nan=True)
    assert not np.isfinite(got).all() and np.isfinite(got).any()


def _hist(rng, W, H, bits, fill):
    hits = np.floor(np.exp(rng.uniform(0.0, 5.0, (H, W)))) * (rng.uniform(0, 1, (H, W)) < fill)
    b = np.zeros((H, W, 5))
    b[:, :, 3] = b[:, :, 4] = hits * 255
    for k in range(3):
        b[:, :, k] = np.floor(hits * rng.uniform(0, 255, (H, W)))
    return b if bits == 64 else b.astype(np.uint32)


def _both(prod, b, bits, widths, coefs, mfi=None, start=None):
    H, W = b.shape[:2]
    out = []
    for f in (prod.lib().fl3h_density_estimate, prod.lib().fl3h_density_estimate_production):
        acc = np.zeros((H, W, 4), dtype=np.float64 if bits == 64 else np.float32)
        if start is not None:
            acc[:] = start
        assert f(b.ctypes.data_as(ctypes.c_void_p), W, H, bits, 1, 1068.0, 1.0 / 2000.0, 0.4,
                 len(widths) - 1, len(widths) - 1 if mfi is None else mfi, coefs.shape[1], len(widths),
                 widths.ctypes.data_as(ctypes.c_void_p), coefs.ctypes.data_as(ctypes.c_void_p),
                 acc.ctypes.data_as(ctypes.c_void_p)) == 0, prod.last_error()
        out.append(acc)
    return out


def _compare(prod, bits, W, H, bank, fill, mfi=None):
    widths, coefs = bank
    rng = np.random.default_rng(W * 1000 + H)
    b = _hist(rng, W, H, bits, fill)
    start = rng.uniform(0.0, 2.0, (H, W, 4)).astype(np.float64 if bits == 64 else np.float32)
    exact, got = _both(prod, b, bits, widths, coefs, mfi, start)
    half = int(np.ceil(widths.max())) - 1
    terms = min((2 * half + 1) ** 2, W * H)
    eps = 2.0 ** (-53 if bits == 64 else -24)
    # per term the exact mode rounds its sum once (and in double three factors),
    # production its sum once and four factors (two of them to float at bits 33)
    tol = (2 * terms + 8) * eps * 1.01
    np.testing.assert_allclose(got, exact, rtol=tol, atol=0)
    if fill == 1.0:
        assert (got > start).any()


@pytest.mark.parametrize("curve", [0.25, 0.4, 0.5, 0.9, 1.0, 3.0, 5.5])
def test_kernel_index_beyond_100_hits(prod, curve):
    """Kernel 100 + floor((hits - 100)^curve): every kernel reaches its own cell
    alone, with a coefficient that tells its index.  Counts at and beside the
    powers' integers and anywhere between.  (At an integer itself either side of
    it is right: the power there is a matter of its last bit.)"""
    nf = 1000
    widths, coefs = np.full(nf, 0.9), np.arange(1.0, nf + 1)[:, None].copy()
    rng = np.random.default_rng(7)
    x = np.arange(1, 920) ** (1 / curve)
    x = np.concatenate([x, x * (1 + 1e-7), x * (1 - 1e-7), x * (1 + 3e-6), x * (1 - 3e-6), np.round(x),
                        np.exp(rng.uniform(-3, np.log(1000.0) / curve, 20000))])
    W = 128
    x = np.resize(x, (len(x) // W, W))
    b = np.zeros(x.shape + (5,))
    b[..., 3] = 255.0
    b[..., 4] = 255.0 * (x + 100)
    fsel = b[..., 4] / 255.0
    acc = np.zeros(x.shape + (4,))
    assert prod.lib().fl3h_density_estimate(
        b.ctypes.data_as(ctypes.c_void_p), W, x.shape[0], 64, 1, 1068.0, 1.0 / 2000.0, curve, 2**31 - 1, nf - 1, 1, nf,
        widths.ctypes.data_as(ctypes.c_void_p), coefs.ctypes.data_as(ctypes.c_void_p),
        acc.ctypes.data_as(ctypes.c_void_p)) == 0, prod.last_error()
    got = np.rint(acc[..., 3] / (1068.0 * np.log(1.0 + 255.0 / 2000.0))).astype(int) - 1
    p = (fsel - 100) ** curve
    ok = (fsel > 100) & (fsel < 2**31 - 1)
    lo, hi = (np.minimum(100 + np.floor(p * f), nf - 1) for f in (1 - 1e-12, 1 + 1e-12))
    assert ok.sum() > 10000
    assert ((got >= lo) & (got <= hi))[ok].all()
