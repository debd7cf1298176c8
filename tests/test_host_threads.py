"""The lock that keeps a render's device calls together.  All CPU; no GPU calls
beyond the attempt to find one."""
import ctypes
import threading

import pytest

from flam3_amd import genome as G


def _device_call(lib, done):
    """A device call of another thread that needs no device: nothing is deferred."""
    n = ctypes.c_double()
    lib.fl3d_deferred_badvals(ctypes.byref(n))
    done.set()


def test_device_calls_of_other_threads_wait(prod_lib):
    done = threading.Event()
    prod_lib.fl3d_hold()
    prod_lib.fl3d_hold()
    t = threading.Thread(target=_device_call, args=(prod_lib, done))
    t.start()
    assert not done.wait(0.2)
    prod_lib.fl3d_release()
    assert not done.wait(0.2)
    prod_lib.fl3d_release()
    assert done.wait(30)
    t.join()


@pytest.mark.parametrize("many", [False, True])
def test_renders_let_go_whatever_their_end(prod_lib, many):
    """Without a device the render fails at its first device call; with one it
    ends well.  Neither keeps the lock."""
    import flam3_amd
    g = G.synthetic_preview(3, size=32, quality=5.0)
    try:
        flam3_amd.render_many([{"genomes": g}]) if many else flam3_amd.render(g)
    except RuntimeError:
        pass
    done = threading.Event()
    threading.Thread(target=_device_call, args=(prod_lib, done), daemon=True).start()
    assert done.wait(30)
