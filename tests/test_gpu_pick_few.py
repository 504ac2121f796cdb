"""The species of sparse passes (many cells, few slots each) against the
general pick: a hadron's draws depend on its cell and its number in it only, so
a part of a surface that is small enough for the general kernel gets the same
hadrons, bit for bit, as in the sparse pass over the whole surface.  Species
lists of one to eight species per lane (up to 512), some of zero yield; cells
without slots, and cells with more slots than a wave draws at a time."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu

N = 140001
PART = 20011


@pytest.fixture(scope="module")
def species():
    return tables.species_arrays(1)


@pytest.fixture(scope="module")
def cells(species):
    c, _ = synth.viscous_lrf(N, species, seed=12, target_hadrons=0.6 * N)
    c = c.copy()
    c[5:PART:997, 4:8] *= 300.0
    c[7:PART:31, 4:8] *= -1.0   # no yields
    return c


def _list(ctx, cells, **opts):
    ctx.set_surface_lrf(cells)
    ctx.sample(1, seed=5, hydro_mode=2, **opts)
    assert ctx.stats().n_range_errors == 0
    h = ctx.hadrons()
    return h[h["pid"] != 0]


def _words(h):
    w = np.ascontiguousarray(h).view(np.int32).reshape(-1, 10)
    return w[np.lexsort(w.T)]


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("ns", [1, 2, 64, 65, 190, 200, 257, 0, 400, 449, 512])
def test_sparse_pass_picks_as_the_general_one(species, cells, ns, precision):
    n = species["mass"].size
    idx = np.arange(ns or n) % n
    sp = {k: np.asarray(species[k])[idx] for k in ("pid", "mass", "g", "B", "S", "Q", "sign")}
    if ns > 2:
        sp["g"][3::7] = 0
        sp["g"][-5:] = 0
    ctx = iss_amd.Context(0)
    ctx.set_species(sp)
    ctx.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=tables.read_kind11(1))
    whole = _list(ctx, cells, precision=precision)
    part = _list(ctx, cells[:PART], precision=precision)
    key = np.isin(whole["x"], cells[:PART, 1]) & np.isin(whole["y"], cells[:PART, 2])
    assert part.size > 1000 or ns <= 2
    assert np.array_equal(_words(whole[key]), _words(part))
    ctx.close()
