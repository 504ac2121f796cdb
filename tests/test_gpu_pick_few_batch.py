"""The species of sparse batched rounds (many cells, few slots each, one- and
several-round batches, both row precisions) against the general pick: a
surface at the head of a batch gets the same hadrons, bit for bit, in a batch
of few surfaces, which takes the general kernel.  Cell counts follow the
device's CUs, so that the whole batch takes the sparse kernel."""
import numpy as np
import pytest
import torch

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu

HEAD = 3


@pytest.fixture(scope="module")
def surfaces():
    sp = tables.species_arrays(1)
    n = 16 * 32 * torch.cuda.get_device_properties(0).multi_processor_count + 12345
    c, _ = synth.viscous_lrf(n, sp, seed=12, target_hadrons=0.3 * n)
    c = c.copy()
    c[5:4000:997, 4:8] *= 300.0   # (more slots than a wave draws at a time)
    c[7:4000:31, 4:8] *= -1.0     # no yields
    cuts = [0, 1001, 2005, 4000, 4001] + list(range(20000, n, 30000)) + [n]
    return sp, [c[a:b] for a, b in zip(cuts, cuts[1:])]


def _head(ctx, cells, events, precision):
    ctx.set_surfaces_lrf(cells)
    ctx.sample_batch(events, seed=5, events_per_round=2, precision=precision)
    seg, ev = ctx.batch_layout()
    h = ctx.hadrons()
    return seg, [np.ascontiguousarray(h[o:o + n]).view(np.int32) for o, n in seg[:, :HEAD].reshape(-1, 2)], ev[:, :HEAD]


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("ns", [1, 7, 64, 65, 200, 257, 0, 400, 512])
def test_sparse_rounds_pick_as_the_general_ones(surfaces, ns, precision):
    species, cells = surfaces
    n = species["mass"].size
    idx = np.arange(ns or n) % n
    sp = {k: np.asarray(species[k])[idx] for k in ("pid", "mass", "g", "B", "S", "Q", "sign")}
    if ns > 7:
        sp["g"][3::7] = 0
        sp["g"][-5:] = 0
    ctx = iss_amd.Context(0)
    ctx.set_species(sp)
    ctx.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=tables.read_kind11(1))
    # a short list has a fraction of the yields: more area for a like number of hadrons
    ctx.set_surface_lrf(np.concatenate(cells[:HEAD]))
    area = np.float32(0.3 * 4000 / ctx.compute_yields(precision=precision).sum())
    scaled = [c.copy() for c in cells]
    for c in scaled:
        c[:, 4:8] *= area
    events = np.full(len(cells), 2, np.int32)
    events[0] = 5
    whole, h_whole, ev_whole = _head(ctx, scaled, events, precision)
    assert whole[0, :, 1].sum() < 1.9 * sum(len(c) for c in cells)   # (sparse: up to two slots a cell)
    part, h_part, ev_part = _head(ctx, scaled[:HEAD], events[:HEAD], precision)
    assert part[0, :, 1].sum() > 1000
    assert np.array_equal(ev_whole, ev_part)
    for a, b in zip(h_whole, h_part):
        assert np.array_equal(a, b)
    ctx.close()
