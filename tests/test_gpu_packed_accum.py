"""The packed accumulation of tile-sorted records (partial sums of the work
items of a full tile, alpha as a multiple of the count where the palettes
allow it) against per-sample atomics: the same integers, so the same image."""
import numpy as np
import pytest

from flam3_amd import genome as G

pytestmark = pytest.mark.gpu


class _Shaded(G.Genome):
    """Palette entries of one alpha below 1, of differing alphas, or of values
    that bytes don't hold."""
    shade = "bytes"

    def to_struct(self):
        gp = super().to_struct()
        for i in range(256):
            c = gp.contents.palette[i].color
            if self.shade == "veiled":
                c[3] = 0.3
            elif self.shade == "alpha":
                c[3] = (i % 7) / 6.0
            elif self.shade == "bright":
                for k in range(3):
                    c[k] *= 3.0
        return gp


def _shaded(g, shade):
    g.__class__ = _Shaded
    g.shade = shade
    g.estimator_radius = 0.0
    return g


@pytest.mark.parametrize("shade", ["bytes", "veiled", "alpha", "bright"])
@pytest.mark.parametrize("size,quality,walkers,chunk", [
    ((64, 64), 300, 1024, 1024 * 700),      # one tile, many items
    ((64, 65), 260, 256, 256 * 64),         # items of exactly a chunk's records and a ragged last tile
    ((640, 481), 4, 1024, 0),               # sparse tiles of one item
    ((333, 217), 90, 2048, 2048 * 2000)])   # both, over chunks
def test_packed_accumulation_equals_atomics(prod, shade, size, quality, walkers, chunk):
    g = _shaded(G.synthetic_small(seed=40, width=size[0], height=size[1], quality=quality), shade)
    a, _ = prod.render(g, seed="acc", nwalkers=walkers, deposit=1, nchan=4, transp=1)
    b, _ = prod.render(g, seed="acc", nwalkers=walkers, deposit=2, chunk_samples=chunk, nchan=4, transp=1)
    assert np.array_equal(a, b)
    assert a[..., :3].mean() > 1.0


@pytest.mark.parametrize("shades", [("bytes", "bytes", "bytes"), ("bytes", "veiled", "alpha"),
                                    ("bytes", "bright", "veiled")])
def test_renders_of_several_palettes_together(prod, shades):
    items = [{"genomes": _shaded(G.synthetic_preview(60 + k, size=s, quality=60), sh), "seed": "p%d" % k, "nchan": 4,
              "transp": 1} for k, (s, sh) in enumerate(zip((64, 200, 129), shades))]
    for it, (img, _) in zip(items, prod.render_many(items)):
        want, _ = prod.render(it["genomes"], seed=it["seed"], nchan=4, transp=1, deposit=1)
        assert np.array_equal(img, want), it["seed"]


@pytest.mark.parametrize("quality", [4112, 4113])
@pytest.mark.parametrize("opacity", [1.0, 0.5, 1.5])
def test_direct_deposits_on_both_sides_of_their_bound(prod, quality, opacity):
    """Channels added in pairs, without reading them back, while 255 times the
    samples stays below 2^32 and no delta passes 255 (4112 x 64 x 64 samples
    and visibility 1); one by one beyond."""
    g = _shaded(G.synthetic_small(seed=41, width=64, height=64, quality=quality), "alpha")
    g.xforms[1].opacity = opacity
    a, sa = prod.render(g, seed="pairs", deposit=1, nchan=4, transp=1)
    b, sb = prod.render(g, seed="pairs", deposit=2, nchan=4, transp=1)
    assert sa["num_iters"] == sb["num_iters"] == quality * 64 * 64
    assert np.array_equal(a, b)


@pytest.mark.parametrize("opacity", [1.0, 0.5])
@pytest.mark.parametrize("width,height,quality", [
    (40, 30, 3), (1000, 1024, 3), (1040, 1024, 3), (2040, 2040, 2), (2060, 2060, 2),      # about 256, 1024 tiles
    (3060, 4070, 1), (3100, 4096, 1), (4560, 4570, 0.5), (4640, 4640, 0.5), (5760, 5760, 0.4)])   # 3072, 5120, 8192
def test_sort_by_the_number_of_tiles(prod, width, height, quality, opacity):
    """Records of 4 and (an opacity below 1, or 2^24 cells) 8 bytes, sorted by
    each form's workgroups, the last of a chunk partly filled."""
    g = _shaded(G.synthetic_small(seed=43, width=width, height=height, quality=quality), "bytes")
    g.xforms[1].opacity = opacity
    a, _ = prod.render(g, seed="sort", deposit=1)
    b, _ = prod.render(g, seed="sort", deposit=2, chunk_samples=700001)
    assert np.array_equal(a, b)
    assert a.any()


@pytest.mark.parametrize("quality", [7.99, 8])
@pytest.mark.parametrize("opacity", [1.0, 0.5])
def test_small_renders_on_both_sides_of_the_sorted_deposit(prod, quality, opacity):
    """The library's own choice of deposit around 32768 samples."""
    g = _shaded(G.synthetic_small(seed=44, width=64, height=64, quality=quality), "alpha")
    g.xforms[1].opacity = opacity
    a, sa = prod.render(g, seed="line", nchan=4, transp=1)
    b, sb = prod.render(g, seed="line", deposit=1, nchan=4, transp=1)
    assert (sa["badvals"], sa["num_iters"]) == (sb["badvals"], sb["num_iters"])
    assert np.array_equal(a, b)
