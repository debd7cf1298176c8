"""Renders of several walker launches whose counters the host reads once at the
end: bad-value counts over repeated batches."""
import numpy as np
import pytest

from flam3_amd import genome as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("passes", [1, 2])
def test_bad_values_of_a_repeated_batch_count_once(prod, passes):
    """Two launches of 9e6 samples a batch, nearly all in one cell, with atomics.
    No sum can reach 2^32 in the first (16.8e6 samples of 255), whose counters
    are read at the end; the second saturates, so the batch is repeated.  One
    draw in ten gives a bad value, so a plotted step meets p / (1 - p) = 1 / 9 of
    them on average (its retries stop at four: 1e-5 off).  The 64 walkers of a
    wavefront share a draw: of 2.8e5 draws 3.1e4 are bad, a spread of 0.6%."""
    point = G.Xform(weight=0.9, coefs=(0.0,) * 6, variations={"linear": 1.0})
    bad = G.Xform(weight=0.1, coefs=(0.0, 0.0, 0.0, 0.0, 1e12, 0.0), variations={"linear": 1.0})
    g = G.Genome(width=8, height=8, scale=4.0, quality=passes * 18e6 / 64, palette=np.full((256, 3), 255.0),
                 estimator_radius=0.0, xforms=[point, bad], passes=passes, temporal_samples=2)
    _, st = prod.render(g, seed="bad", deposit=1, temporal_batch=1)
    assert st["num_iters"] >= 18e6 * passes - 1000
    assert st["badvals"] / st["num_iters"] == pytest.approx(1 / 9, rel=0.02)
