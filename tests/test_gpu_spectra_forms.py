"""The FP64 eta_s-integrated spectra (linear and quadratic forms of the lab
momentum) against the rapidity-resolved ones (rest-frame contraction), which
are held to the oracle elsewhere: with every cell at eta_s = 0 the integrated
spectrum is sum_k w_k dN(y = -eta_k).

Both are FP64; the forms differ by the rounding of terms up to (u^0 cosh y)^2
~ 1e4 times the result, about 1e-12, so the bar is 1e-10 of the row maximum."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables
from tests import neos22_table

pytestmark = pytest.mark.gpu

TOL = 1e-10
DELTAF = {
    "ideal": dict(shear=0, bulk=0),
    "shear": dict(shear=1, bulk=0),
    "rta": dict(shear=1, bulk=1, bulk_kind=1),
    "osu14": dict(shear=1, bulk=1, bulk_kind=11),
    "ce": dict(shear=1, bulk=1, bulk_kind=21),
    "mom22": dict(shear=1, bulk=1, bulk_kind=20),
    "diffusion": dict(shear=1, bulk=1, bulk_kind=11, diffusion=1),
}


def _context(name, cells):
    ctx = iss_amd.Context(0)
    ctx.set_species(tables.species_arrays(1))
    kw = dict(DELTAF[name])
    kind = kw.get("bulk_kind")
    if kind == 11:
        kw["k11"] = tables.read_kind11(1)
    if kind == 21:
        kw["neos"] = tables.read_neos(21, 1)
    if kind == 20:
        kw["neos"] = neos22_table.table()
    if kw.get("diffusion"):
        kw["qmu_table"] = tables.read_qmu_table()
    ctx.set_deltaf(**kw)
    ctx.set_surface_lrf(cells)
    return ctx


def _cells(n, seed, charged=True):
    c, _ = synth.viscous_lrf(n, tables.species_arrays(1), seed=seed, diffusion=0.1)
    ut = np.sqrt(1.0 + c[:, 9] ** 2 + c[:, 10] ** 2)
    c[:, 3], c[:, 8], c[:, 11] = 0.0, ut, 0.0
    if charged:
        c[:, 17], c[:, 18] = -0.03, 0.01
    return c


def _check(ctx, idx, pT, phi, eta, w, **kw):
    got = ctx.spectra(idx, pT, phi, eta, w, mode=0, precision=64, **kw)
    ref = ctx.spectra(idx, pT, phi, -eta, mode=1, precision=64, **kw)
    ref = np.einsum("k,skij->sij", w, ref)
    scale = np.abs(ref).max(axis=-1, keepdims=True)
    assert np.all(np.abs(got - ref) <= TOL * scale)  # (rows of exact zeros included)


@pytest.mark.parametrize("name", list(DELTAF))
@pytest.mark.parametrize("restrict", [0, 1])
def test_every_deltaf_form(name, restrict):
    rng = np.random.default_rng(3)
    ctx = _context(name, _cells(9, 4))
    _check(ctx, np.array([0, 3, 20, 21, 150]), np.linspace(0.05, 3.0, 7), rng.uniform(0, 6.28, 11),
           np.linspace(-3.0, 3.0, 31), rng.uniform(0.5, 1.0, 31), restrict_deltaf=restrict, deltaf_max_ratio=0.7)
    ctx.close()


@pytest.mark.parametrize("n_pT,n_phi,n_eta,n_cells", [
    (1, 1, 1, 1), (5, 51, 63, 2), (16, 16, 64, 7), (1, 257, 65, 3), (3, 171, 129, 33), (15, 48, 81, 130)])
def test_grid_remainders(n_pT, n_phi, n_eta, n_cells):
    rng = np.random.default_rng(n_eta)
    ctx = _context("osu14", _cells(n_cells, n_cells))
    _check(ctx, np.array([1, 17]), np.linspace(0.1, 2.5, n_pT), rng.uniform(0, 6.28, n_phi),
           np.linspace(-3.5, 3.5, n_eta), rng.uniform(0.5, 1.0, n_eta))
    ctx.close()


def test_far_rapidities_and_positive_only():
    """|eta| = 20 (an exponent of 1e9: no occupancy, no NaN) and dropped
    negative contributions, on space-like cells."""
    c = _cells(40, 6)
    c[:, 5:8] *= 6.0
    ctx = _context("osu14", c)
    eta = np.array([-20.0, -8.0, -0.5, 0.0, 0.7, 20.0])
    w = np.array([1.0, 0.5, 0.3, 0.2, 0.3, 1.0])
    idx, pT, phi = np.array([0, 18]), np.array([0.0, 0.4, 2.0]), np.linspace(0, 6.0, 9)
    _check(ctx, idx, pT, phi, eta, w)
    out = ctx.spectra(idx, pT, phi, eta, w, mode=0, precision=64, use_pos_dN_only=1)
    assert np.all(np.isfinite(out)) and np.all(out >= 0)
    ctx.close()


@pytest.mark.parametrize("name", ["ideal", "rta", "osu14", "mom22", "diffusion"])
@pytest.mark.parametrize("potentials", ["none", "B", "BQ", "S"])
@pytest.mark.parametrize("precision", [32, 64])
def test_species_evaluated_together_equal_species_alone(name, potentials, precision):
    """One call for species that share masses and charges against one call
    per species: the same sums up to the grouping of cells into chunks (FP64
    sums of 60 cells: 1e-13)."""
    c = _cells(60, 9)
    c[:, 16] *= "B" in potentials
    c[:, 17] *= "S" in potentials
    c[-1, 18] = 0.02 if "Q" in potentials else 0.0   # (one cell alone has mu_Q)
    c[:-1, 18] = 0.0
    ctx = _context(name, c)
    sp = tables.species_arrays(1)
    idx = np.array([0, 1, 2, 3, 4, 5, 6, 0, 16, 17, 18, 19, 21, 22, 40, 41, 42, 43])
    assert len(set(zip(sp["mass"][idx], sp["B"][idx]))) < idx.size
    pT, phi, eta, w = np.linspace(0.1, 2.0, 4), np.linspace(0, 5.5, 6), np.linspace(-2, 2, 9), np.full(9, 0.5)
    for mode in (0, 1):
        together = ctx.spectra(idx, pT, phi, eta, w, mode=mode, precision=precision)
        alone = np.stack([ctx.spectra([i], pT, phi, eta, w, mode=mode, precision=precision)[0] for i in idx])
        scale = np.abs(alone).max(axis=-1, keepdims=True)
        assert np.all(np.abs(together - alone) <= 1e-13 * scale)
    ctx.close()
