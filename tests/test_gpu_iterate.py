"""fl3h_iterate with few walkers (one per wavefront) against the same walkers
among many (one per lane): the same points, random states and bad-value
counts, bit for bit."""
import ctypes

import numpy as np
import pytest

from flam3_amd import abi
from flam3_amd import genome as G

pytestmark = pytest.mark.gpu

LANES = 4097   # walkers: one more than run one per wavefront


def _classic():
    """Every classic variation, in xforms of one to seven of them."""
    rng = np.random.default_rng(1)
    names = list(abi.VARIATION_NAMES[:14])
    return [G._mixed_xform(rng, names, k, -1.0, 1.0) for k in range(1, 8)]


def _all(seed):
    """Variations of the whole library (parameters at their defaults)."""
    rng = np.random.default_rng(seed)
    names = [n for n in abi.VARIATION_NAMES]
    return [G._mixed_xform(rng, names, 12, -1.0, 1.0) for _ in range(6)]


def _genome(kind):
    if kind == "final_opacity":
        g = G.synthetic_1080p(seed=5, width=64, height=36)
        g.final.opacity = 0.4
        return g
    if kind == "xaos":
        return G.synthetic_8k(seed=6, width=64, height=36)
    if kind == "bad_values":
        g = G.synthetic_small(seed=7, width=64, height=48)
        g.xforms[0].coefs = (1e7, 0.0, 0.0, 1e7, 0.0, 0.0)
        return g
    if kind == "one_xform":
        xs = _classic()[:1]
    elif kind == "classic":
        xs = _classic()
        for x in xs[::2]:
            x.post = (0.5, 0.1, -0.2, 0.7, 0.05, -0.1)
    elif kind == "preblur":
        xs = _classic()
        for x in xs:
            x.variations["pre_blur"] = 0.3
    else:
        xs = _all(int(kind[3:]))
    return G.Genome(width=64, height=48, scale=16.0, xforms=xs)


def _run(L, g, walkers, n, fuse):
    arr, owned = G.genome_array([g])
    gp = ctypes.cast(ctypes.addressof(arr), ctypes.POINTER(abi.flam3_genome))
    try:
        # the bounding box prepares the genome as the reference's callers do
        f = abi.flam3_frame()
        L.fl3h_init_frame(ctypes.byref(f), b"prepare")
        box = (ctypes.c_double * 4)()
        L.fl3h_estimate_bounding_box(gp, 0.01, 8, box, ctypes.byref(box, 16), ctypes.byref(f.rc))
        nstd = len(g.xforms)
        table = np.tile(((np.arange(16384) * nstd) // 16384).astype(np.uint16), nstd + 1)
        rc = (abi.randctx * walkers)()
        for w in range(walkers):
            L.fl3h_init_frame(ctypes.byref(f), b"walker-%d" % w)
            ctypes.memmove(ctypes.byref(rc[w]), ctypes.byref(f.rc), ctypes.sizeof(f.rc))
        pts = np.zeros((walkers, n, 4))
        pts[:, 0] = np.random.default_rng(8).uniform(-1.0, 1.0, (LANES, 4))[:walkers]
        bad = np.zeros(walkers, np.int32)
        assert L.fl3h_iterate(gp, n, fuse, pts.ctypes.data, table.ctypes.data, rc, walkers, bad.ctypes.data) == 0
        state = [bytes(rc[w]) for w in range(min(walkers, 65))]
        return pts[:65].tobytes(), state, bad[:65].tolist()
    finally:
        for p in owned:
            G.free_struct(p)


@pytest.mark.parametrize("kind", ["classic", "one_xform", "preblur", "xaos", "final_opacity", "bad_values", "all1",
                                  "all2", "all3"])
def test_few_walkers_equal_the_same_among_many(prod, kind):
    L = prod.lib()
    L.fl3h_estimate_bounding_box.argtypes = [ctypes.c_void_p, ctypes.c_double, ctypes.c_int] + [ctypes.c_void_p] * 3
    L.fl3h_estimate_bounding_box.restype = ctypes.c_int
    g = _genome(kind)
    few, many = _run(L, g, 65, 40, 20), _run(L, g, LANES, 40, 20)
    assert few[2] == many[2]
    assert few[1] == many[1]
    assert few[0] == many[0]
