"""The plain trial kernel's lane groups: a hadron's draws depend on its cell
and its number in it only, so the cells of a surface get the same hadrons, bit
for bit, when they are sampled alone (few hadrons, up to 64 lanes each) and
when they are sampled with many others (one lane each until the list ends)."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu

N = 6000


@pytest.fixture(scope="module", params=[(5000, 2), (5000, 1), (3, 2)], ids=["3d", "boost_invariant", "few_trials"])
def whole(request):
    max_trials, mode = request.param
    sp = tables.species_arrays(1)
    cells, _ = synth.viscous_lrf(N, sp, seed=9, target_hadrons=0.2 * N)
    ctx = iss_amd.Context(0)
    ctx.set_species(sp)
    ctx.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=tables.read_kind11(1))
    opts = dict(seed=77, max_trials=max_trials, hydro_mode=mode, y_LB=-1.0, y_RB=1.0)
    yield ctx, cells, opts, _list(ctx, cells, opts)
    ctx.close()


def _list(ctx, cells, opts):
    ctx.set_surface_lrf(cells)
    n = ctx.sample(100, **opts)
    h = ctx.hadrons()
    assert h.size == n
    st = ctx.stats()
    h = h[h["pid"] != 0]
    assert n - h.size == st.n_failed and st.n_range_errors == 0
    assert st.n_inner >= st.n_trials >= h.size
    return h


def _sorted_words(h):
    w = np.ascontiguousarray(h).view(np.int32).reshape(-1, 10)
    return w[np.lexsort(w.T)]


@pytest.mark.parametrize("n", [1, 2, 3, 5, 31, 64, 65, 257, 1000, 3001])
def test_cells_alone_get_the_same_hadrons(whole, n):
    ctx, cells, opts, everything = whole
    sub = cells[:n]
    got = _list(ctx, sub, opts)
    key = np.isin(everything["x"], sub[:, 1]) & np.isin(everything["y"], sub[:, 2])
    want = everything[key]
    assert got.size == want.size
    assert np.array_equal(_sorted_words(got), _sorted_words(want))
