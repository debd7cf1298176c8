"""Histograms of more than 2^13 tiles in 32-bit cells at full-size chunks of
records: the atomics' image, in the memory that records and tiles need."""
import ctypes

import numpy as np
import pytest

from flam3_amd import genome as G

pytestmark = pytest.mark.gpu


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("fade", [False, True])
def test_banded_bits33_at_full_chunks(prod, fade):
    """5800 x 5800 cells, 3.03e8 samples: a chunk of 2^28 records and the rest.
    Integer sums, so the image equals the per-sample atomics' exactly.  Records
    (8 bytes, two buffers and the sorted ones: 7.2 GB with the allocations'
    eighth), histogram and accumulator (1.4 GB) and partial sums (0.4 GB) leave
    room below 16 GB."""
    g = G.synthetic_small(seed=82, width=5800, height=5800, quality=9)
    g.estimator_radius = 0.0
    if fade:
        g.xforms[1].opacity = 0.5
    before = _free_bytes()
    b, sb = prod.render(g, seed="band", deposit=2)
    assert before - _free_bytes() < 16e9
    a, sa = prod.render(g, seed="band", deposit=1)
    assert sa["num_iters"] == sb["num_iters"] and sa["num_iters"] > 1 << 28
    assert sa["badvals"] == sb["badvals"]
    assert np.array_equal(a, b)
    assert a.mean() > 1.0
