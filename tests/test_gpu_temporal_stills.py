"""Stills with temporal samples, which share one set of selection breakpoints,
against the same genome as two equal control points, whose samples each have
their own."""
import copy

import numpy as np
import pytest

from flam3_amd import genome as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("xaos", [False, True])
@pytest.mark.parametrize("samples,passes", [(2, 1), (5, 1), (5, 3)])
def test_still_equals_two_equal_control_points(prod, samples, passes, xaos, many):
    """A temporal filter of no width puts every sample at time 0, the first
    control point itself, which linear affines and an RGB palette blend give
    back exactly."""
    rng = np.random.default_rng(8)
    xs = [G._mixed_xform(rng, G.WORKLOAD_VARS, 2, -1.0, 1.0) for _ in range(7)]
    if xaos:
        for x in xs:
            x.chaos = [float(c) for c in rng.uniform(0.1, 2.0, 7)]
    g = G.Genome(width=64, height=48, scale=16.0, quality=20.0, passes=passes, temporal_samples=samples,
                 temporal_filter_width=0.0, interpolation_type="linear", palette_interpolation="rgb",
                 palette=np.floor(G.hsv_palette(rng)), xforms=xs)
    two = [g, copy.deepcopy(g)]
    two[1].time = 1.0
    if many:
        img, st = prod.render_many([{"genomes": g, "seed": "t"}])[0]
    else:
        img, st = prod.render(g, seed="t")
    want, ws = prod.render(two, seed="t", time=0.0)
    assert (st["num_iters"], st["badvals"]) == (ws["num_iters"], ws["badvals"])
    assert np.array_equal(img, want)
    assert img.max() > 0
