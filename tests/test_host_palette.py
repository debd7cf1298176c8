"""Palettes a Genome takes: anything whose first 256 entries have three numbers.
All CPU."""
import numpy as np
import pytest

from flam3_amd import genome as G

ROWS = np.random.default_rng(3).uniform(0.0, 255.0, (256, 4))


def _colours(prod, palette):
    g = G.Genome(width=8, height=8, palette=palette, xforms=[G.Xform(weight=1.0, variations={"linear": 1.0})])
    gp = g.to_struct()
    try:
        return np.array([[e.index] + list(e.color) for e in gp.contents.palette])
    finally:
        G.free_struct(gp)


@pytest.mark.parametrize("name,palette", [
    ("array", ROWS[:, :3]), ("rgba", ROWS), ("float32", ROWS.astype(np.float32)), ("bytes", ROWS.astype(np.uint8)),
    ("longer", np.vstack([ROWS, ROWS[:9]])), ("lists", ROWS.tolist()),
    ("tuples", [tuple(r[:3 + i % 2]) for i, r in enumerate(ROWS)]),
    ("rows_of_differing_ends", [list(r[:3]) for r in ROWS] + [[1.0]]), ("by_index", dict(enumerate(ROWS)))])
def test_entries(prod, name, palette):
    got = _colours(prod, palette)
    want = np.array([[float(i), *(float(palette[i][k]) / 255.0 for k in range(3)), 1.0] for i in range(256)])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("palette", [ROWS[:255], ROWS[:, :1], ROWS[:, :2], ROWS[:, :1].tolist(), ROWS[:255].tolist()])
def test_too_few_numbers(prod, palette):
    with pytest.raises(IndexError):
        _colours(prod, palette)


@pytest.mark.parametrize("palette", [(ROWS + 1j).tolist(), ROWS.reshape(256, 4, 1)[:, :, [0, 0]]])
def test_no_numbers(prod, palette):
    with pytest.raises(TypeError):
        _colours(prod, palette)
