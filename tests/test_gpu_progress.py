"""The progress callback of a render of several launches follows the device."""
import ctypes
import time

import numpy as np
import pytest

from flam3_amd import abi
from flam3_amd import genome as G
from flam3_amd._lib import fl3h_render_opts

pytestmark = pytest.mark.gpu


def _calls(prod, g, deposit, stop=None):
    """Render g, a launch per temporal sample; the callback's times, and those of
    the render's start and end."""
    PROG = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_double, ctypes.c_int, ctypes.c_double)
    at = []

    def cb(param, pct, stage, eta):
        at.append((time.perf_counter(), pct))
        return int(len(at) == stop)

    cfun = PROG(cb)
    arr, owned = G.genome_array([g])
    try:
        f = prod.make_frame(ctypes.addressof(arr), 1, progress=cfun)
        img = np.zeros((g.height, g.width, 3), dtype=np.uint8)
        opts = fl3h_render_opts(0, 0, deposit, 0, 1)
        t0 = time.perf_counter()
        rc = prod.lib().fl3h_render(ctypes.byref(f), img.ctypes.data_as(ctypes.c_void_p), 0, 3, 0,
                                    ctypes.byref(abi.stat_struct()), ctypes.byref(opts))
        t1 = time.perf_counter()
        assert rc == 0
        return t0, at, t1
    finally:
        for gp in owned:
            G.free_struct(gp)


@pytest.mark.parametrize("deposit,quality", [(2, 60000), (1, 200)])
def test_callback_waits_for_the_launches_before_it(prod, deposit, quality):
    """Three equal launches of some 10 ms (sorted deposits) or 4 ms (atomics that
    cannot saturate).  A sample's callback comes before its launch is made, the
    launch before it made after the one's before: so the third callback finds one
    launch done, a third of the device's work, and an abort there waits for no
    other."""
    g = G.synthetic_small(seed=76, width=256, height=256, quality=quality)
    g.estimator_radius = 0.0
    g.temporal_samples = 3
    _calls(prod, g, deposit)
    t0, at, t1 = _calls(prod, g, deposit)
    assert [round(p) for _, p in at] == [0, 33, 67]
    assert at[2][0] - at[1][0] > 0.15 * (t1 - at[1][0])
    _, at, t2 = _calls(prod, g, deposit, stop=3)
    assert len(at) == 3
    assert t2 - at[2][0] < 0.15 * (t1 - t0)
