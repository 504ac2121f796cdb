"""Batches of many surfaces and of many rounds: the layout's invariants where
the event trees are taken some rounds at a time and where the surfaces are
more than a workgroup."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu


def _batch(S, cells_each, hadrons, events, R, **kw):
    sp = tables.species_arrays(1)
    ctx = iss_amd.Context(0)
    ctx.set_species(sp)
    ctx.set_deltaf(shear=1, bulk=0)
    c, _ = synth.viscous_lrf(S * cells_each, sp, seed=S, target_hadrons=hadrons, bulk=False, shear=True)
    ctx.set_surfaces_lrf([c[k * cells_each:(k + 1) * cells_each] for k in range(S)])
    n = ctx.sample_batch(events, seed=21, events_per_round=R, **kw)
    seg, ev = ctx.batch_layout()
    rounds = -(-int(events.max()) // R)
    assert seg.shape == (rounds, S, 2) and ev.shape == (rounds, S, R)
    # blocks follow one another, each the sum of its events, none past a surface's last
    assert np.array_equal(seg[..., 0].ravel(), np.concatenate([[0], np.cumsum(seg[..., 1].ravel())])[:-1])
    assert seg[..., 1].sum() == n
    assert np.array_equal(ev.sum(axis=2), seg[..., 1])
    left = np.clip(events[None] - R * np.arange(rounds)[:, None], 0, R)
    assert not ev[np.arange(R)[None, None] >= left[..., None]].any()
    assert not seg[left == 0, 1].any()
    # every surface's hadrons, and all: Poisson with the yields' mean
    _, per = ctx.compute_yields(precision=32, per_cell=True)
    mean = events * per.astype(np.float64).sum(axis=1).reshape(S, cells_each).sum(axis=1)
    got = seg[..., 1].sum(axis=0)
    assert np.all(np.abs(got - mean) < 7 * np.sqrt(mean) + 12) and abs(n - mean.sum()) < 6 * np.sqrt(mean.sum())
    return ctx, seg, ev


def test_event_sizes_of_many_rounds():
    """1000 surfaces in rounds of 16 events: 64 MB hold the trees of 524
    rounds; 1100 rounds take three passes, the last of 52.  Events of a round
    are alike: their places in it have the same hadrons over all rounds, to
    six standard deviations."""
    S, R, rounds = 1000, 16, 1100
    events = np.full(S, 3, np.int32)
    events[0], events[1] = R * rounds, R * 530 + 7
    ctx, seg, ev = _batch(S, 1, 5.0 * S, events, R)
    place = ev[:, 0, :].sum(axis=0)
    mean = seg[:, 0, 1].sum() / R
    assert np.abs(place - mean).max() < 6 * np.sqrt(mean)
    ctx.close()


@pytest.mark.parametrize("S", [255, 256, 257, 1000, 2049])
@pytest.mark.parametrize("use_graph", [0, 1])
def test_many_surfaces(S, use_graph):
    """Three rounds of surfaces with 1 to 5 events; rounds replayed and rounds
    launched give the same list."""
    events = (1 + np.arange(S) % 5).astype(np.int32)
    ctx, seg, ev = _batch(S, 2, 3.0 * S, events, 2, use_graph=use_graph)
    h = ctx.hadrons()
    other = ctx.sample_batch(events, seed=21, events_per_round=2, use_graph=1 - use_graph)
    assert other == h.size and np.array_equal(ctx.hadrons(), h)
    ctx.close()
