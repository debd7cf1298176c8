"""Renders with a side of 2^24 cells and more: no records, whose 24-bit product
of the width and the row would put the second row's points in the first."""
import numpy as np
import pytest

from flam3_amd import genome as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("many", [False, True])
def test_rows_of_more_than_2_24_cells(prod, many):
    """Two rows of 2^24 + 8 cells, 1.7e5 samples, enough for a smaller histogram's
    to be sorted: points in both rows, and the atomics' image."""
    W = (1 << 24) + 8
    g = G.Genome(width=W, height=2, scale=1.0, quality=0.005, palette=np.full((256, 3), 255.0), estimator_radius=0.0,
                 brightness=1e6,
                 xforms=[G.Xform(weight=0.5, coefs=(0.1, 0.0, 0.0, 0.1, 2.0 * k, s), variations={"linear": 1.0})
                         for k, s in ((-2, -0.45), (2, 0.45))])
    if many:
        img, st = prod.render_many([{"genomes": g, "seed": "long"}])[0]
    else:
        img, st = prod.render(g, seed="long", deposit=0)
    want, ws = prod.render(g, seed="long", deposit=1)
    assert st["num_iters"] == ws["num_iters"] > 32768
    assert want[0].any() and want[1].any()
    assert np.array_equal(img, want)
