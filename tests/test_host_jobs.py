"""What the host prepares for each temporal sample, by its short ways against
its general ones: breakpoints of the xform selection without the table, and
genomes between control points that share a segment."""
import ctypes

import numpy as np
import pytest

from flam3_amd import abi
from flam3_amd import genome as G

GRAIN = 16384


def _lib(prod):
    L = prod.lib()
    L.fl3_create_xform_distrib.restype = ctypes.c_void_p
    L.fl3_create_xform_distrib.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    L.fl3_distrib_breakpoints.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    L.fl3_xform_starts.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    L.fl3_segment_open.restype = ctypes.c_void_p
    L.fl3_segment_open.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_double]
    L.fl3_segment_close.argtypes = [ctypes.c_void_p]
    L.fl3_interpolate.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_double, ctypes.c_double, ctypes.c_void_p]
    L.fl3_interpolate_in.argtypes = [ctypes.c_void_p] + L.fl3_interpolate.argtypes
    return L


WEIGHTS = {
    "any": lambda r, n: r.uniform(0.0, 1.0, n),
    "equal": lambda r, n: np.ones(n),
    "quarters": lambda r, n: 0.25 * r.integers(0, 4, n) + (np.arange(n) == 0),
    "spread": lambda r, n: np.exp(r.uniform(-30.0, 30.0, n)),
    "sparse": lambda r, n: r.uniform(0.0, 1.0, n) * (r.uniform(0, 1, n) < 0.3) + (np.arange(n) == n - 1),
    "last_places": lambda r, n: (1.0 + r.integers(0, 8, n) * 2.0 ** -51) * 2.0 ** r.integers(0, 5, n),
    "tiny": lambda r, n: r.uniform(0.0, 1.0, n) * 1e-290,
    "huge": lambda r, n: r.uniform(0.0, 1.0, n) * 1e250,
}


@pytest.mark.parametrize("kind", list(WEIGHTS))
@pytest.mark.parametrize("xaos", [False, True])
def test_breakpoints_equal_the_tables(prod, kind, xaos):
    L = _lib(prod)
    for n in (1, 2, 3, 7, 12, 40):
        for seed in range(4):
            rng = np.random.default_rng(1000 * n + seed)
            w = WEIGHTS[kind](rng, n)
            xs = [G._mixed_xform(rng, ["linear"], 1, -1.0, 1.0) for _ in range(n)]
            for x, v in zip(xs, w):
                x.weight = float(v)
                if xaos:
                    x.chaos = [float(c) for c in rng.integers(0, 3, n) * 0.5 + 0.01]
            gp = G.Genome(width=64, height=48, scale=16.0, xforms=xs).to_struct()
            try:
                rows = ctypes.c_int()
                got = np.full(((n + 1), n), -1, np.int32)
                want = got.copy()
                assert L.fl3_xform_starts(gp, got.ctypes.data, ctypes.byref(rows)) == 0
                assert rows.value == (n + 1 if gp.contents.chaos_enable else 1)
                table = L.fl3_create_xform_distrib(gp, None)
                L.fl3_distrib_breakpoints(table, rows.value, n, want.ctypes.data)
                ctypes.CDLL(None).free(ctypes.c_void_p(table))
                assert np.array_equal(got, want), (n, seed)
            finally:
                G.free_struct(gp)


@pytest.mark.parametrize("weights", [(0.0, 0.0), (0.5, -0.1)])
def test_weights_without_a_table_are_refused(prod, weights):
    L = _lib(prod)
    rng = np.random.default_rng(2)
    xs = [G._mixed_xform(rng, ["linear"], 1, -1.0, 1.0) for _ in weights]
    for x, v in zip(xs, weights):
        x.weight = v
    gp = G.Genome(width=64, height=48, scale=16.0, xforms=xs).to_struct()
    starts = np.zeros(6, np.int32)
    assert L.fl3_xform_starts(gp, starts.ctypes.data, None) != 0
    G.free_struct(gp)


def _bytes(g):
    """The genome's and its xforms' bytes, without pointers."""
    b = bytearray(ctypes.string_at(ctypes.addressof(g), ctypes.sizeof(g)))
    for f in ("xform", "chaos", "edits"):
        if hasattr(abi.flam3_genome, f):
            o = getattr(abi.flam3_genome, f).offset
            b[o:o + 8] = bytes(8)
    n = ctypes.sizeof(abi.flam3_xform) * g.num_xforms
    return bytes(b), ctypes.string_at(ctypes.cast(g.xform, ctypes.c_void_p).value, n)


@pytest.mark.parametrize("kind", ["linear", "log", "old", "older"])
@pytest.mark.parametrize("curve", ["linear", "smooth"])
@pytest.mark.parametrize("palette", ["hsv", "sweep", "rgb", "hsv_circular"])
def test_shared_segment_equals_interpolation_alone(prod, kind, curve, palette):
    L = _lib(prod)
    gs = []
    for k in range(4):
        rng = np.random.default_rng(50 + k)
        xs = [G._mixed_xform(rng, list(abi.VARIATION_NAMES), 4, -1.2, 1.2) for _ in range(2 + k % 3)]
        g = G.Genome(width=64, height=48, scale=16.0, xforms=xs, palette=G.hsv_palette(rng))
        if k % 2:
            g.final = G._mixed_xform(rng, ["linear", "blob"], 2, -1.0, 1.0)
        g.time, g.interpolation_type, g.interpolation, g.palette_interpolation = 10.0 * k, kind, curve, palette
        gs.append(g)
    arr, owned = G.genome_array(gs)
    try:
        for at in (-1.0, 4.0, 15.0, 30.0):
            seg = L.fl3_segment_open(ctypes.byref(arr), 4, at)
            assert seg
            a, b = abi.flam3_genome(), abi.flam3_genome()
            for t in (0.0, 4.5, 10.0, 12.5, 19.9, 25.0, 31.0):   # its own segment's times and others'
                assert L.fl3_interpolate(ctypes.byref(arr), 4, t, 0.2, ctypes.byref(a)) == 0
                assert L.fl3_interpolate_in(seg, ctypes.byref(arr), 4, t, 0.2, ctypes.byref(b)) == 0
                assert _bytes(a) == _bytes(b), (at, t)
            L.fl3h_genome_clear(ctypes.byref(a))
            L.fl3h_genome_clear(ctypes.byref(b))
            L.fl3_segment_close(seg)
        assert not L.fl3_segment_open(ctypes.byref(arr), 1, 0.0)
    finally:
        for p in owned:
            G.free_struct(p)
