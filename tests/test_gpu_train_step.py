"""The training step's workgroup sums at batch sizes around its loops (one
workgroup, fewer and more than the 32 gradients loaded together, a ragged
last workgroup), against the sums of single-workgroup evaluations: a sample's
loss, inputs and output gradient do not depend on its workgroup (exact), and
the gradient of all samples is the FP32 sum of the workgroups' (n workgroups
of O(1) terms: n 6e-8 of the summed magnitudes)."""
import numpy as np
import pytest

import iss_amd
from iss_amd import synth, tables

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    sp = tables.species_arrays(1)
    cells, _ = synth.viscous_lrf(300, sp, seed=12, target_hadrons=300.0)
    c = iss_amd.Context(0)
    c.set_species(sp)
    c.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=tables.read_kind11(1), fermion_cdf2_quirk=0)
    c.set_surface_lrf(cells)
    c.mlp_init(3)
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 64, 65, 31 * 64, 32 * 64, 33 * 64 + 7, 71 * 64])
def test_gradient_is_the_sum_over_workgroups(ctx, n):
    rng = np.random.default_rng(n)
    cell, spec = rng.integers(0, 300, n), rng.integers(0, 60, n)
    whole = ctx.mlp_eval(cell, spec)
    parts = [ctx.mlp_eval(cell[i:i + 64], spec[i:i + 64]) for i in range(0, n, 64)]
    for k in ("loss", "dz", "x"):
        assert np.array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    g = np.stack([p["grad"].astype(np.float64) for p in parts])
    assert np.all(np.abs(whole["grad"] - g.sum(axis=0)) <= len(parts) * 6e-8 * np.abs(g).sum(axis=0) + 1e-30)


def test_trained_weights_are_the_weights_sampled_with(ctx):
    """The step rewrites the packed weights: uploading the trained parameters
    (which packs them afresh) changes nothing."""
    ctx.sample(400, seed=4)
    ctx.mlp_collect(100_000)
    ctx.mlp_init(3)
    ctx.mlp_train(batch=256, steps=7, lr=3e-3, seed=1)
    cell, spec = np.arange(200), np.arange(200) % 40
    a = ctx.mlp_eval(cell, spec)
    ctx.mlp_set_params(ctx.mlp_get_params())
    b = ctx.mlp_eval(cell, spec)
    for k in ("loss", "dz", "grad"):
        assert np.array_equal(a[k], b[k])
