"""The exclusive scan at the sizes where its launches change (one tile, tiles
that add the sums before them, a separate scan of the sums), seen through the
event sizes: counts of a uniform multinomial, so that a wrong offset of a tile
shows as a negative or far too large event at its edge."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu

TILE = 2048
DIRECT = 1024


@pytest.fixture(scope="module")
def ctx():
    sp = tables.species_arrays(1)
    cells, _ = synth.viscous_lrf(3, sp, seed=4, target_hadrons=1.5)
    c = iss_amd.Context(0)
    c.set_species(sp)
    c.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=tables.read_kind11(1))
    c.set_surface_lrf(cells)
    yield c
    c.close()


@pytest.mark.parametrize("events", [1, 2, TILE - 1, TILE, TILE + 1, 2 * TILE + 1, DIRECT * TILE - 1, DIRECT * TILE,
                                    DIRECT * TILE + 1, DIRECT * TILE + 5 * TILE])
def test_event_sizes_at_scan_edges(ctx, events):
    n = ctx.sample(events, seed=events)
    sizes = np.asarray(ctx.event_counts())
    assert sizes.size == events and sizes.sum() == n
    # Poisson of mean n / events < 4: beyond 40 has probability < 1e-25
    assert sizes.min() >= 0 and (events < 100 or sizes.max() < 40)
