"""Rapidity-resolved spectra of enough species and cells for the kernel that
takes a point's rapidities together (two waves per CU), against the one that
boosts every point by itself, as test_gpu_spectra_rapidity.py; and species that
share an integrand in calls large enough to ask for it."""
import numpy as np
import pytest
import torch

from iss_amd import tables
from tests.test_gpu_spectra_forms import DELTAF, _cells as _still_cells, _context
from tests.test_gpu_spectra_rapidity import _cells

pytestmark = pytest.mark.gpu


def _compare(name, n_pT, n_phi, n_y, n_cells, precision, **kw):
    chunks, waves = -(-n_y // 6), -(-n_pT * n_phi // 128)
    ns = -(-2 * torch.cuda.get_device_properties(0).multi_processor_count // (chunks * waves * -(-n_cells // 8)))
    assert ns <= 321 and 5 * n_pT * n_phi >= 192 * -(-n_pT * n_phi // 64)
    ctx = _context(name, _cells(n_cells, 7))
    rng = np.random.default_rng(n_pT * 1000 + n_phi)
    idx, y = np.arange(ns), np.linspace(-1.5, 1.5, n_y)
    pT, phi = np.linspace(0.05, 3.0, n_pT), rng.uniform(0, 6.28, n_phi)
    got = ctx.spectra(idx, pT, phi, y, mode=1, precision=precision, **kw)
    ref = np.empty_like(got)
    for i in range(n_pT):
        for j in range(0, n_phi, 32):
            ref[:, :, i:i + 1, j:j + 32] = ctx.spectra(idx, pT[i:i + 1], phi[j:j + 32], y, mode=1, precision=precision,
                                                       **kw)
    scale = np.abs(ref).max(axis=-1, keepdims=True)
    assert np.all(np.abs(got - ref) <= (1e-10 if precision == 64 else 1e-5) * scale)
    ctx.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", list(DELTAF))
@pytest.mark.parametrize("positive", [0, 1])
def test_every_deltaf_form(name, positive, precision):
    _compare(name, 4, 24, 7, 19, precision, use_pos_dN_only=positive, deltaf_max_ratio=0.7)


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("n_pT,n_phi,n_y,n_cells", [
    (1, 39, 3, 17), (2, 64, 5, 16), (3, 43, 6, 9), (4, 48, 7, 8), (2, 97, 12, 33), (1, 255, 13, 40), (3, 86, 19, 5)])
def test_grid_edges(n_pT, n_phi, n_y, n_cells, precision):
    _compare("osu14", n_pT, n_phi, n_y, n_cells, precision)


@pytest.mark.parametrize("name", ["ideal", "rta", "osu14", "mom22", "diffusion"])
@pytest.mark.parametrize("potentials", ["none", "B", "BQ", "S"])
@pytest.mark.parametrize("precision", [32, 64])
def test_species_evaluated_together_equal_species_alone(name, potentials, precision):
    """600 cells: the sums differ by the grouping of their terms, 600 2^-53
    of the sum of magnitudes at most: 1e-12."""
    c = _still_cells(600, 9)
    c[:, 16] *= "B" in potentials
    c[:, 17] *= "S" in potentials
    c[-1, 18] = 0.02 if "Q" in potentials else 0.0   # (one cell alone has mu_Q)
    c[:-1, 18] = 0.0
    ctx = _context(name, c)
    sp = tables.species_arrays(1)
    idx = np.array([0, 1, 2, 3, 4, 5, 6, 0, 16, 17, 18, 19, 21, 22, 40, 41, 42, 43])
    spared = idx.size - len(set(zip(sp["mass"][idx], sp["sign"][idx])))
    pT, phi, eta, w = np.linspace(0.1, 2.0, 15), np.linspace(0, 5.5, 40), np.linspace(-2, 2, 9), np.full(9, 0.5)
    assert spared * 600.0 * 600 * 9 > 1e7
    for mode in (0, 1):
        together = ctx.spectra(idx, pT, phi, eta, w, mode=mode, precision=precision)
        alone = np.stack([ctx.spectra([i], pT, phi, eta, w, mode=mode, precision=precision)[0] for i in idx])
        scale = np.abs(alone).max(axis=-1, keepdims=True)
        assert np.all(np.abs(together - alone) <= 1e-12 * scale)
    ctx.close()
