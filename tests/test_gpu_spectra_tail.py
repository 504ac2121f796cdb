"""FP64 integrated spectra where the occupancy runs out of the double range
(E / T up to 750): against the rapidity-resolved kernel, whose exponential and
reciprocal are the library's.  The exponent (E - mu) / T log2(e) of up to 1021
has rounding 2^-53 of it, so values agree to 1e-12; beyond 1024 there are none."""
import numpy as np
import pytest

from iss_amd import synth, tables
from tests.test_gpu_spectra_forms import _context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["ideal", "rta", "osu14", "diffusion"])
def test_tail_of_the_double_range(name):
    sp = tables.species_arrays(1)
    c, _ = synth.viscous_lrf(1, sp, seed=8, diffusion=0.1)
    c[:, 3] = 0.0
    c[:, 8:12] = [1.0, 0.0, 0.0, 0.0]   # at rest: E = mT
    idx = [0, 2, int(np.argmax(sp["mass"]))]
    ctx = _context(name, c)
    x = np.array([3.0, 500.0, 990.0, 999.0, 1001.0, 1010.0, 1019.0])
    phi = np.array([0.3, 2.0, 4.4])
    for i in idx:
        B, S, Q = (float(sp[k][i]) for k in "BSQ")
        E = x * np.log(2.0) * c[0, 13] + B * c[0, 16] + S * c[0, 17] + Q * c[0, 18]
        ok = E > sp["mass"][i]
        pT = np.sqrt(E[ok] ** 2 - sp["mass"][i] ** 2)
        got = ctx.spectra([i], pT, phi, [0.0], [1.0], mode=0, precision=64, deltaf_max_ratio=0.5)[0]
        ref = ctx.spectra([i], pT, phi, [0.0], mode=1, precision=64, deltaf_max_ratio=0.5)[0, 0]
        assert np.all(ref != 0) and np.all(np.abs(got - ref) <= 1e-12 * np.abs(ref))
        far = ctx.spectra([i], [200.0], phi, [0.0], [1.0], mode=0, precision=64)
        assert np.all(far == 0)
    ctx.close()
