"""What the host layer does around its kernels, seen through a stand-in for
the HIP runtime (tests/fake_hip.cpp): no GPU, no kernel runs.  Every test is a
program of its own, since the stand-in has to be loaded before the library."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, numpy as np
fake = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
for f in ("fake_launched", "fake_copies", "fake_host_allocs", "fake_largest"):
    getattr(fake, f).restype = C.c_int64
fake.fake_known.argtypes = [C.c_void_p, C.c_int64, C.c_int]
import iss_amd

def launched(part):
    # how often a kernel was launched; workgroups and threads of the last time
    groups, threads = C.c_int64(), C.c_int64()
    n = fake.fake_launched(part.encode(), C.byref(groups), C.byref(threads))
    return n, groups.value, threads.value

def context():
    ctx = iss_amd.Context(0)
    ctx.set_species(dict(pid=[211, -211, 2212], mass=[0.14, 0.14, 0.938], g=[1, 1, 2], B=[0, 0, 1], S=[0, 0, 0],
                         Q=[1, -1, 1], sign=[-1, -1, 1]))
    return ctx

def read_list(ctx, nbytes, known=0):
    # sets a list of that size, reads it back: the read-back's blocking copies and pinned allocations
    words = np.arange(nbytes // 4, dtype=np.int32)
    ctx.set_hadrons([words.size // 10], words.view(iss_amd.HADRON_DTYPE))
    got = np.zeros_like(words)
    fake.fake_known(got.ctypes.data, nbytes, known)
    fake.fake_reset()
    assert ctx.lib.iss_get_hadrons(ctx.h, got.ctypes.data_as(C.c_void_p), words.size // 10) == 0
    assert np.array_equal(got, words)
    return fake.fake_copies(), fake.fake_host_allocs()

def cells(n):
    c = np.zeros((n, 28), np.float32)
    c[:, 8], c[:, 13] = 1.0, 0.15
    return c
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    so = os.path.join(str(tmp_path_factory.mktemp("fake")), "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", so, os.path.join(ROOT, "tests", "fake_hip.cpp")],
                   check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(so=so) + body], cwd=ROOT, capture_output=True, text=True,
                           timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


@pytest.mark.parametrize("change", ["ctx.set_surface_lrf(cells(900))", "ctx.set_deltaf(shear=1)"])
def test_trial_words_are_not_used_after_a_failed_change(program, change):
    """Whichever allocation, copy or wait fails in a change of surface or delta
    f, a pass that the caller runs all the same does not take the words (nor
    the yields) of what was there before."""
    program(f"""
for n in range(1, 40):
    ctx = context()
    ctx.set_surface_lrf(cells(100))
    ctx.sample(1)
    assert launched("k_trial_cells")[0] > 0
    ctx.sample(1)
    fake.fake_reset()
    ctx.sample(1)
    assert launched("k_trial_cells")[0] == 0 and launched("k_yield_rows")[0] == 0
    fake.fake_reset()
    fake.fake_fail(n, 0)
    try:
        {change}
        failed = False
    except iss_amd.ISSError:
        failed = True
    fake.fake_fail(0, 0)
    ctx.sample(1)
    assert ctx.num_cells() == 0 or (launched("k_trial_cells")[0] > 0 and launched("k_yield_rows")[0] > 0), n
    ctx.close()
    if not failed:
        break
assert n > 1
""")


def test_lists_for_memory_that_the_runtime_knows_take_its_copy(program):
    """Page-locked (1) and device (2) destinations: one copy of the runtime,
    no staging; pageable ones go through the ring."""
    program("""
for known in (1, 2):
    assert read_list(context(), 100 << 20, known) == (1, 0)
assert read_list(context(), 100 << 20) == (0, 1)
""")


def test_lists_come_back_where_pinned_memory_runs_out(program):
    """The ring's slots cannot be had: the runtime's copy, now and at the next
    list, then the ring once they can."""
    program("""
ctx = context()
for _ in range(2):
    fake.fake_fail(0, 1)
    assert read_list(ctx, 100 << 20) == (1, 1)
assert read_list(ctx, 100 << 20) == (0, 1)
""")


def test_short_lists_take_the_ring_once_they_repay_its_slots(program):
    """Lists of 5 MB: the runtime's copy until they have come to 12 MB; one of
    13 MB takes the ring at once, and short ones after it use its slots."""
    program("""
ctx = context()
MB5, MB13, MB30 = (n * (1 << 20) // 40 * 40 for n in (5, 13, 30))
assert [read_list(ctx, MB5) for _ in range(4)] == [(1, 0)] * 2 + [(0, 1), (0, 0)]
ctx = context()
assert [read_list(ctx, n) for n in (MB13, MB5, MB13)] == [(0, 1), (0, 0), (0, 0)]
assert [read_list(ctx, n) for n in (MB30, MB5, MB30)] == [(0, 1), (0, 0), (0, 0)]
""")


def test_event_trees_of_many_rounds_stay_small(program):
    """1000 surfaces, 20,000 events of one of them: 1250 rounds of 16 events.
    The largest buffer is the event sizes themselves (uint32 [rounds][S][R])."""
    program("""
ctx = context()
ctx.set_surfaces_lrf([cells(1)] * 1000)
events = np.ones(1000, np.int32)
events[0] = 20000
fake.fake_reset()
ctx.sample_batch(events, events_per_round=16)
assert 0 < fake.fake_largest() <= 4 * 1250 * 1000 * 16
assert launched("k_batch_multi_leaves")[0] > 1
ctx.sample_batch(np.full(1000, 16, np.int32), events_per_round=16)
fake.fake_reset()
ctx.sample_batch(np.full(1000, 16, np.int32), events_per_round=16)
assert launched("k_batch_multi_leaves")[0] == 1
""")


def test_kernels_of_many_surfaces_fit_them(program):
    """The kernels over surfaces: at most 64 surfaces a workgroup of a round's
    roots, and no 16-wave workgroups for the sums of a few cells."""
    program("""
for S, n_cells, want in ((1, 2, (1, 256)), (64, 2, (1, 256)), (65, 2, (2, 256)), (1000, 2, (16, 256)), (3, 2000, (1, 1024))):
    ctx = context()
    ctx.set_surfaces_lrf([cells(n_cells)] * S)
    ctx.sample_batch(np.full(S, 3, np.int32), events_per_round=2)
    assert (launched("k_batch_roots")[1], launched("k_batch_lambda")[2]) == want, (S, want)
    ctx.close()
""")


def test_small_spectra_launch_only_what_they_repay(program):
    """Species that could share an integrand: the surface is asked for its
    potentials, and the shared sums spread, only where that spares evaluations
    worth the question.  Few waves: the general kernel of the rapidities."""
    program("""
def spectra(n_cells, idx, n_pT, n_phi, n_y, mode=1):
    ctx = context()
    ctx.set_surface_lrf(cells(n_cells))
    fake.fake_reset()
    ctx.spectra(idx, np.linspace(0.1, 2.0, n_pT), np.linspace(0, 6.0, n_phi), np.linspace(-2, 2, n_y), np.ones(n_y),
                mode=mode, precision=64)
    ctx.close()
    return [launched(k)[0] for k in ("k_mu_used", "k_spectra_spread", "k_spectra_points", "k_spectra_y")]

for mode, kernel in ((0, [0, 0]), (1, [1, 0])):
    assert spectra(300, [0, 1, 2], 1, 10, 1, mode) == [0, 0] + kernel
assert spectra(20000, [0, 2], 15, 48, 11) == [0, 0, 0, 1]       # (two masses)
assert spectra(20000, [0, 1, 2], 15, 48, 11) == [1, 1, 0, 1]
assert spectra(300, [0], 7, 16, 11) == [0, 0, 1, 0]
assert spectra(300, [0], 7, 16, 2) == [0, 0, 0, 1]
assert spectra(2040, [0], 7, 16, 11) == [0, 0, 1, 0]            # (510 waves)
assert spectra(2048, [0], 7, 16, 11) == [0, 0, 0, 1]
""")


def test_sparse_rounds_take_the_sparse_pick(program):
    """512 cells a CU and at most two slots a cell; else the general pick."""
    program("""
for n_cells, want in ((131071, [0, 1]), (131072, [1, 0])):
    ctx = context()
    ctx.set_surfaces_lrf([cells(n_cells)])
    fake.fake_reset()
    ctx.sample_batch(np.full(1, 2, np.int32), events_per_round=2, use_graph=1)
    few, all_picks = launched("k_pick_few")[0], launched("k_pick")[0]
    assert [few, all_picks - few] == want, (n_cells, few, all_picks)
    ctx.close()
""")
