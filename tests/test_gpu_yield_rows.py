"""The yield rows' sharing of work: a cell's yields, its total and the counts
drawn from it do not depend on how many cells the surface has (tiles of 64
cells, shares that split a tile between waves), nor a species' yield on the
other species of the list (segments of 8 or 16, light species one at a time).

Same operations per item: rows agree to a few roundings (FP64 1e-13, FP32
2e-6); species totals are FP64 sums of the rows (1e-12); the counts drawn with
one seed agree exactly (a cell total off by an ulp moves none of these few
thousand draws, one off by a lost or doubled segment moves many)."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 129, 1000, 2049, 5000]
RTOL = {64: 1e-13, 32: 2e-6}


@pytest.fixture(scope="module")
def species():
    return tables.species_arrays(1)


@pytest.fixture(scope="module")
def cells(species):
    c, _ = synth.viscous_lrf(SIZES[-1], species, seed=21, target_hadrons=4000.0)
    c[:, 17], c[:, 18] = -0.02, 0.005
    return c


def _context(sp, cells):
    ctx = iss_amd.Context(0)
    ctx.set_species(sp)
    ctx.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=tables.read_kind11(1))
    ctx.set_surface_lrf(cells)
    return ctx


def _subset(sp, idx):
    return {k: np.asarray(sp[k])[idx] for k in ("pid", "mass", "g", "B", "S", "Q", "sign")}


@pytest.mark.parametrize("precision", [32, 64])
def test_rows_totals_and_counts_by_surface_size(species, cells, precision):
    big = _context(species, cells)
    tot, rows = big.compute_yields(precision=precision, per_cell=True)
    assert np.allclose(tot, rows.sum(axis=0, dtype=np.float64), rtol=1e-12)
    big.sample(3, seed=5, precision=precision)
    h = big.hadrons()
    key = {tuple(x): i for i, x in enumerate(cells[:, 1:3].tolist())}
    counts = np.bincount([key[(x, y)] for x, y in zip(h["x"].tolist(), h["y"].tolist())], minlength=len(cells))
    big.close()
    for n in SIZES[:-1]:
        ctx = _context(species, cells[:n])
        t, r = ctx.compute_yields(precision=precision, per_cell=True)
        assert np.allclose(r, rows[:n], rtol=RTOL[precision], atol=0)
        assert np.allclose(t, rows[:n].sum(axis=0, dtype=np.float64), rtol=max(1e-12, 1e-2 * RTOL[precision]))
        assert ctx.sample(3, seed=5, precision=precision) == counts[:n].sum()
        ctx.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("pick", [[0], [7], [8], list(range(8)), list(range(9)), list(range(2, 19)), list(range(5, 45)),
                                  list(range(8, 321))], ids=str)
def test_rows_by_species_list(species, cells, precision, pick):
    c = cells[:200]
    full = _context(species, c)
    tot, rows = full.compute_yields(precision=precision, per_cell=True)
    full.close()
    ctx = _context(_subset(species, pick), c)
    t, r = ctx.compute_yields(precision=precision, per_cell=True)
    assert np.allclose(r, rows[:, pick], rtol=RTOL[precision], atol=0)
    assert np.allclose(t, tot[pick], rtol=max(1e-12, RTOL[precision]))
    ctx.close()


@pytest.mark.parametrize("precision", [32, 64])
def test_charges_outside_the_fugacity_rows_take_the_general_series(species, cells, precision):
    """A species of charge 3 (outside the staged fugacity factors) switches the
    whole pass; the other species' yields stay."""
    c = cells[:130]
    full = _context(species, c)
    _, rows = full.compute_yields(precision=precision, per_cell=True)
    full.close()
    sp = {k: np.array(v) for k, v in _subset(species, np.arange(40)).items()}
    sp["Q"][39] = 3
    ctx = _context(sp, c)
    _, r = ctx.compute_yields(precision=precision, per_cell=True)
    assert np.allclose(r[:, :39], rows[:, :39], rtol=1e-11 if precision == 64 else 1e-5, atol=0)
    ctx.close()
