"""Yields of unusual cells, FP64 and FP32 rows: potentials that are not
numbers leave the whole cell without yields and its neighbours alone; cells so
cold (0.045 to 0.05 GeV) that every species has one term while its K arguments
are still inside the staged rows, against the oracle."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables
from tests import oracle_binding as ob

pytestmark = pytest.mark.gpu


def _context(sp):
    ctx = iss_amd.Context(0)
    ctx.set_species(sp)
    ctx.set_deltaf(shear=1, bulk=1, bulk_kind=1)
    return ctx


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("field", [16, 17, 18])
def test_potential_that_is_not_a_number(field, precision):
    sp = tables.species_arrays(1)
    c, _ = synth.viscous_lrf(130, sp, seed=3)
    ctx = _context(sp)
    ctx.set_surface_lrf(c)
    _, ref = ctx.compute_yields(precision=precision, per_cell=True)
    bad = c.copy()
    bad[[0, 63, 64, 101], field] = np.nan
    ctx.set_surface_lrf(bad)
    tot, got = ctx.compute_yields(precision=precision, per_cell=True)
    keep = ~np.isnan(bad[:, field])
    assert not got[~keep].any()
    assert np.array_equal(got[keep], ref[keep])
    assert np.allclose(tot, got.astype(np.float64).sum(axis=0), rtol=1e-12)
    ctx.close()


@pytest.mark.parametrize("precision", [32, 64])
def test_cold_cells_of_one_term(precision):
    """The heaviest species of 2.3 GeV at 0.0455 GeV: m / T = 50.5, below the
    51.7 of the staged rows.  0.05 GeV (as a float, just above) has ten terms,
    the float below it one."""
    sp = tables.species_arrays(1)
    sp = {k: np.asarray(v)[np.asarray(sp["mass"]) < 2.3] for k, v in sp.items()
          if k in ("pid", "mass", "g", "B", "S", "Q", "sign")}
    c, _ = synth.viscous_lrf(200, sp, seed=5, bulk=False)
    c[:, 13] = np.linspace(0.0455, 0.0499, 200)
    c[7, 13] = np.nextafter(np.float32(0.05), np.float32(0))
    c[:, 16:19] = [0.05, 0.01, -0.01]
    ctx = _context(sp)
    ctx.set_surface_lrf(c)
    _, got = ctx.compute_yields(precision=precision, per_cell=True)
    orc = ob.Oracle(afterburner=1, shear=1, bulk=1, bulk_kind=1)
    orc.set_cells_lrf(c)
    ref = orc.yields()[:, np.asarray(tables.species_arrays(1)["mass"]) < 2.3]
    # (the bars of test_gpu_yields.py)
    assert np.all(np.abs(got - ref) <= (1e-6 if precision == 64 else 1e-5) * np.abs(ref) + 1e-30)
    ctx.close()
