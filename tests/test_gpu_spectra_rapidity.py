"""Rapidity-resolved spectra: the kernel that takes the rapidities of a (pT,
phi) point together against the one that boosts every point by itself, which
serves grids of few (pT, phi) points: the same grid whole and in pieces of at
most 32 points.

Both form the rest-frame momentum in FP64 (terms up to ~1e2 times the result,
1e-14) and evaluate the same integrand.  FP64: 1e-10 of the row maximum.  FP32:
a few values round to the neighbouring float, 6e-8 |x| of a term with |x| <=
80: 1e-5 of the row maximum."""
import numpy as np
import pytest

from iss_amd import synth, tables
from tests.test_gpu_spectra_forms import DELTAF, _context

pytestmark = pytest.mark.gpu


def _cells(n, seed):
    c, _ = synth.viscous_lrf(n, tables.species_arrays(1), seed=seed, diffusion=0.1)
    c[:, 17], c[:, 18] = -0.03, 0.01
    return c


def _compare(ctx, n_pT, n_phi, y, precision, **kw):
    rng = np.random.default_rng(n_pT * 1000 + n_phi)
    idx = np.array([0, 3, 20, 150])
    pT, phi = np.linspace(0.05, 3.0, n_pT), rng.uniform(0, 6.28, n_phi)
    got = ctx.spectra(idx, pT, phi, y, mode=1, precision=precision, **kw)
    ref = np.empty_like(got)
    step = min(n_phi, 32)
    for i in range(n_pT):
        for j in range(0, n_phi, step):
            ref[:, :, i:i + 1, j:j + step] = ctx.spectra(idx, pT[i:i + 1], phi[j:j + step], y, mode=1,
                                                         precision=precision, **kw)
    scale = np.abs(ref).max(axis=-1, keepdims=True)
    assert np.all(np.abs(got - ref) <= (1e-10 if precision == 64 else 1e-5) * scale)


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", list(DELTAF))
@pytest.mark.parametrize("positive", [0, 1])
def test_every_deltaf_form(name, positive, precision):
    ctx = _context(name, _cells(19, 4))
    _compare(ctx, 5, 24, np.linspace(-2.0, 2.0, 7), precision, use_pos_dN_only=positive, deltaf_max_ratio=0.7)
    ctx.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("n_pT,n_phi,n_y,n_cells", [
    (1, 39, 3, 2), (1, 64, 1, 1), (1, 77, 2, 7), (2, 64, 5, 8), (3, 43, 6, 9), (4, 48, 7, 17), (2, 97, 12, 33), (1, 255, 13, 40),
    (3, 86, 19, 5)])
def test_grid_edges(n_pT, n_phi, n_y, n_cells, precision):
    ctx = _context("osu14", _cells(n_cells, 7))
    _compare(ctx, n_pT, n_phi, np.linspace(-1.5, 1.5, n_y), precision)
    ctx.close()
