"""Palettes so bright that an accumulation item holds few records: no room for
partial sums, the items add to the histogram with atomics."""
import ctypes

import numpy as np
import pytest

from flam3_amd import genome as G

pytestmark = pytest.mark.gpu


class _Glaring(G.Genome):
    """Colours 1e5 times as bright: entries of up to 2.55e7, items of 168 records."""

    def to_struct(self):
        gp = super().to_struct()
        for i in range(256):
            c = gp.contents.palette[i].color
            for k in range(3):
                c[k] *= 1e5
        return gp


def _square(seed, size, quality):
    """Four maps onto the quarters of a square: every cell is met as often, so
    no cell's sum of `quality` samples' entries nears 2^32."""
    xs = [G.Xform(weight=1.0, color=k / 3.0, coefs=(0.5, 0.0, 0.0, 0.5, x, y), variations={"linear": 1.0})
          for k, (x, y) in enumerate([(-0.5, -0.5), (0.5, -0.5), (-0.5, 0.5), (0.5, 0.5)])]
    return _Glaring(width=size, height=size, scale=size / 2.0, quality=quality, estimator_radius=0.0, xforms=xs,
                    palette=G.hsv_palette(np.random.default_rng(seed)))


def _free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("fade", [False, True])
@pytest.mark.parametrize("size", [64, 500])
def test_glaring_palette_equals_atomics(prod, size, fade):
    g = _square(1, size, 30 if size > 64 else 60)
    if fade:
        for x in g.xforms:
            x.opacity = 0.5
    before = _free_bytes()
    b, sb = prod.render(g, seed="glare", deposit=2, nchan=4, transp=1)
    assert before - _free_bytes() < 2e9
    a, sa = prod.render(g, seed="glare", deposit=1, nchan=4, transp=1)
    assert sa["num_iters"] == sb["num_iters"]
    assert np.array_equal(a, b)
    assert a[..., :3].mean() > 1.0


def test_glaring_palettes_together(prod):
    items = [{"genomes": _square(2 + k, s, 30), "seed": "p%d" % k} for k, s in enumerate((200, 256, 129))]
    for it, (img, _) in zip(items, prod.render_many(items)):
        want, _ = prod.render(it["genomes"], seed=it["seed"], deposit=1)
        assert np.array_equal(img, want), it["seed"]
