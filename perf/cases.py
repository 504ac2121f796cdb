"""Timed cases of the sampler: what a program that samples freeze-out surfaces
has it do, through the Python binding's entry points.

Seven kinds of work:

  yields    per-species totals of a resident surface (compute_yields)
  rows      the yields of every (cell, species) into the caller's device
            buffers (compute_yields_noalloc)
  spectra   smooth Cooper-Frye spectra on a (pT, phi) grid, integrated over
            eta_s (mode 0) or at given rapidities (mode 1)
  sample    one oversampling step of a resident surface: yields, hadrons,
            event sizes and the hadron list on the host
  event     one hydro event from its freeze-out file's cells to the stable
            hadrons: surface, yields, sampling, resonance decays, read-back
  batch     many surfaces of uneven size in one batched pass
  train     the learned proposal's network from its start to trained weights

Sizes follow the configurations of iss_amd/synth.py and bench.py: surfaces
from a few thousand cells (a boost-invariant one) through 200,000 (viscous
3+1D) to a million, 1 to 1000 events per surface, about 0.05 hadrons per cell
and event, the 321 species of the UrQMD list, the reference's quadrature grid
of 15 pT x 48 phi x 81 eta_s.
"""
import ctypes
import functools
import math
import statistics

import numpy as np
import torch

import iss_amd
from iss_amd import synth, tables

HBARC = 0.197327053


# ------------------------------------------------------------------- tables
@functools.lru_cache(None)
def species():
    return tables.species_arrays(1)


@functools.lru_cache(None)
def bins():
    return tables.bin_tables()


@functools.lru_cache(None)
def kind11():
    return tables.read_kind11(1)


@functools.lru_cache(None)
def neos():
    return tables.read_neos(21, 1)


@functools.lru_cache(None)
def qmu():
    return tables.read_qmu_table()


@functools.lru_cache(None)
def eos(kind):
    return tables.read_eos(kind, 1)


@functools.lru_cache(None)
def decays():
    return tables.decay_table(1)


@functools.lru_cache(None)
def thermo_grid():
    return synth.hrg_grid(species(), 0.135, 0.160 + 1e-9, 0.0, 0.45 + 1e-9)


# ----------------------------------------------------------------- surfaces
def lrf_cells(case, seed):
    """Rest-frame cells of a viscous 3+1D surface."""
    n = case["cells"]
    cells, _ = synth.viscous_lrf(n, species(), seed=seed, muB_max=case.get("muB_max", 0.3),
                                 target_hadrons=case.get("per_event", 0.05 * n), grid=thermo_grid(),
                                 bulk=case["deltaf"] != "ideal", shear=case["deltaf"] != "ideal")
    return cells


def binv_cells(n, seed):
    """Lab cells of a boost-invariant ideal surface, tau = 10 fm, radial flow."""
    rng = np.random.default_rng(seed)
    x, y = rng.uniform(-6.0, 6.0, n), rng.uniform(-7.5, 7.5, n)
    r = np.maximum(np.hypot(x, y), 1e-6)
    v = 0.6 * np.tanh(r / 7.0)
    gam = 1.0 / np.sqrt(1.0 - v * v)
    c = np.zeros((n, 34))
    c[:, 0], c[:, 1], c[:, 2], c[:, 4] = 10.0, x, y, 180.0 / n
    c[:, 8], c[:, 9], c[:, 10] = gam, gam * v * x / r, gam * v * y / r
    T = rng.uniform(0.145, 0.155, n)
    e, P, nB = synth.hrg_thermo_fast(T, np.zeros(n), species(), thermo_grid())
    c[:, 12], c[:, 13], c[:, 14] = e, T, P
    return c.astype(np.float32)


def batch_cells(case):
    """Cell counts of a batch's surfaces: log-normal about the median."""
    q = [statistics.NormalDist().inv_cdf((i * 29 % case["surfaces"] + 0.5) / case["surfaces"])
         for i in range(case["surfaces"])]
    return np.clip(np.round(case["median"] * np.exp(q)), 50, 50000).astype(int)


def lab_cells(n, per_event, seed):
    """Lab cells of a viscous 3+1D surface as the hydro code writes them: a
    few per cent with u.dsigma < 0, pi orthogonal to the flow up to rounding,
    a baryon diffusion current."""
    rng = np.random.default_rng(seed)
    c = np.zeros((n, 34))
    tau = rng.uniform(0.8, 12.0, n)
    c[:, 0], c[:, 1], c[:, 2] = tau, rng.uniform(-8, 8, n), rng.uniform(-8, 8, n)
    c[:, 3] = rng.uniform(-4.0, 4.0, n)
    u = np.empty((n, 4))
    u[:, 1], u[:, 2], u[:, 3] = rng.normal(0, 0.8, n), rng.normal(0, 0.8, n), rng.normal(0, 0.3, n)
    u[:, 0] = np.sqrt(1.0 + (u[:, 1:] ** 2).sum(1))
    c[:, 8:12] = u
    T, muB = rng.uniform(0.137, 0.158, n), rng.uniform(0.0, 0.2, n)
    e, P, nB = synth.hrg_thermo_fast(T, muB, species(), thermo_grid())
    c[:, 12], c[:, 13], c[:, 14], c[:, 15], c[:, 16] = e, T, P, nB, muB
    D = np.empty((n, 4))
    D[:, 0] = rng.uniform(0.5, 1.5, n)
    D[:, 1:] = rng.normal(0, 0.25, (n, 3))
    back = rng.uniform(0, 1, n) < 0.1
    D[back, 0] = rng.normal(0, 0.4, back.sum())
    area = per_event / float(np.sum(P / T))
    c[:, 4:7], c[:, 7] = area * D[:, :3] / tau[:, None], area * D[:, 3]
    # pi^{mu nu} and q^mu from the rest frame by the boost to u
    L = np.zeros((n, 4, 4))
    L[:, 0, 0], L[:, 0, 1:], L[:, 1:, 0] = u[:, 0], u[:, 1:], u[:, 1:]
    L[:, 1:, 1:] = np.eye(3) + u[:, 1:, None] * u[:, None, 1:] / (u[:, 0] + 1.0)[:, None, None]
    w = rng.normal(size=(n, 3, 3))
    w = w + w.transpose(0, 2, 1)
    w -= np.trace(w, axis1=1, axis2=2)[:, None, None] * np.eye(3) / 3.0
    w *= (rng.uniform(0, 0.2, n) * (e + P) / np.sqrt((w ** 2).sum((1, 2))))[:, None, None]
    S = np.zeros((n, 4, 4))
    S[:, 1:, 1:] = w
    S = L @ S @ L.transpose(0, 2, 1)
    for k, (a, b) in enumerate([(0, 0), (0, 1), (0, 2), (0, 3), (1, 1), (1, 2), (1, 3), (2, 2), (2, 3), (3, 3)]):
        c[:, 19 + k] = S[:, a, b]
    c[:, 29] = -rng.uniform(0, 0.1, n) * (e + P)
    q = np.zeros((n, 4))
    q[:, 1:] = rng.normal(0, 1, (n, 3))
    q *= (0.1 * np.maximum(nB, 1e-3) / np.linalg.norm(q, axis=1))[:, None]
    c[:, 30:34] = np.einsum("nab,nb->na", L, q)
    return c.astype(np.float32)


def context(case):
    """A context with the species list and the delta f of the case."""
    ctx = iss_amd.Context(0)
    ctx.set_species(species())
    d = case["deltaf"]
    if d == "ideal":
        ctx.set_deltaf(shear=0, bulk=0, fermion_cdf2_quirk=case.get("quirk", 1))
    elif d == "rta":          # the reference's default: shear, relaxation-time bulk
        ctx.set_deltaf(shear=1, bulk=1, bulk_kind=1, fermion_cdf2_quirk=case.get("quirk", 1))
    elif d == "14mom":
        ctx.set_deltaf(shear=1, bulk=1, bulk_kind=11, k11=kind11(), fermion_cdf2_quirk=case.get("quirk", 1))
    elif d == "ce":
        ctx.set_deltaf(shear=1, bulk=1, bulk_kind=21, neos=neos(), fermion_cdf2_quirk=case.get("quirk", 1))
    elif d == "diffusion":
        ctx.set_deltaf(shear=1, bulk=1, bulk_kind=1, diffusion=1, qmu_table=qmu(),
                       fermion_cdf2_quirk=case.get("quirk", 1))
    return ctx


# -------------------------------------------------------------------- cases
def listed():
    return [
        # an event-by-event program's first look at a small boost-invariant
        # surface: thermal yields per unit rapidity, FP64 (the driver's default)
        dict(name="yields_small_fp64", kind="yields", cells=2000, boost_invariant=True, deltaf="ideal", precision=64),
        # every (cell, species) yield of the benchmark's 3+1D surface, FP64, for
        # a program that samples cells itself or checks the sampler
        dict(name="rows_fp64", kind="rows", cells=200003, deltaf="14mom", precision=64),
        # the largest resident surface, FP32 yields (the benchmark's precision)
        dict(name="rows_fp32_large", kind="rows", cells=1000000, deltaf="14mom", precision=32, muB_max=0.45),
        # calculate_vn: spectra of every chosen species on the reference's grid
        dict(name="spectra_all_species", kind="spectra", cells=3001, deltaf="14mom", precision=64, mode=0,
             species=321, pT=15, phi=48, eta=81),
        # identified-hadron spectra (pi, K, p and antiparticles' like) of the
        # benchmark's surface
        dict(name="spectra_identified", kind="spectra", cells=200000, deltaf="14mom", precision=64, mode=0,
             species=3, pT=15, phi=48, eta=81),
        # rapidity-resolved spectra in FP32, a small grid of an ordinary surface
        dict(name="spectra_rapidity_fp32", kind="spectra", cells=20011, deltaf="14mom", precision=32, mode=1,
             species=5, pT=12, phi=24, eta=11),
        # a handful of events of a small boost-invariant surface: latency
        dict(name="sample_small_binv", kind="sample", cells=2000, boost_invariant=True, deltaf="ideal", events=10,
             precision=64, proposal=0, model=30, lcc=0),
        # the benchmark's step with its hadrons read back: ~1e7 of them
        dict(name="sample_large", kind="sample", cells=200000, per_event=10000.0, deltaf="14mom", quirk=0,
             events=1000, precision=32, proposal=0, model=30, lcc=0),
        # heavy oversampling of one surface with the learned proposal
        dict(name="sample_learned", kind="sample", cells=20000, per_event=1000.0, deltaf="14mom", quirk=0,
             events=2000, precision=32, proposal=1, model=30, lcc=0),
        # one hydro event end to end, as the command-line driver runs it:
        # EoS-regulated surface, FP64 yields, 100 oversampled events, decays
        dict(name="event_decays", kind="event", cells=30007, per_event=4000.0, deltaf="ce", eos=14, events=100,
             precision=64, decays=1, model=30, lcc=0),
        # a minimum-bias batch: many surfaces of uneven size in one pass
        dict(name="batch_uneven", kind="batch", surfaces=48, median=6000, deltaf="14mom", quirk=0, events=120,
             precision=32, proposal=0),
        # the learned proposal's training as the driver runs it
        dict(name="train", kind="train", cells=20000, per_event=1000.0, deltaf="14mom", quirk=0, batch=8192,
             steps=100),
    ]


def draw(rng):
    def size(a, b):
        n = int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
        return max(a, min(b, n + rng.choice((-1, 0, 1))))

    kind = rng.choice(("yields", "rows", "rows", "spectra", "spectra", "sample", "sample", "event", "event", "batch",
                       "train"))
    if kind == "yields":
        if rng.random() < 0.4:
            return dict(kind=kind, cells=size(100, 20000), boost_invariant=True, deltaf="ideal",
                        precision=rng.choice((32, 64)))
        return dict(kind=kind, cells=size(100, 200000), deltaf=rng.choice(("ideal", "14mom", "14mom")),
                    precision=rng.choice((32, 64)))
    if kind == "rows":
        p = rng.choice((32, 64))
        return dict(kind=kind, cells=size(500, 800000 if p == 32 else 200000),
                    deltaf=rng.choice(("ideal", "14mom", "14mom")), precision=p)
    if kind == "spectra":
        if rng.random() < 0.3:
            return dict(kind=kind, cells=size(500, 50000), deltaf=rng.choice(("ideal", "14mom")),
                        precision=rng.choice((32, 64)), mode=1, species=rng.choice((1, 3, 5, 11)),
                        pT=rng.randint(5, 15), phi=rng.randint(8, 48), eta=rng.randint(3, 21))
        ns = rng.choice((1, 3, 6, 20, 77, 321))
        return dict(kind=kind, cells=size(100, min(100000, 900000 // ns)), deltaf=rng.choice(("ideal", "14mom")),
                    precision=rng.choice((64, 64, 32)), mode=0, species=ns, pT=rng.randint(7, 15),
                    phi=rng.randint(16, 48), eta=rng.choice((21, 41, 81)))
    if kind == "sample":
        if rng.random() < 0.3:
            return dict(kind=kind, cells=size(200, 10000), boost_invariant=True, deltaf="ideal", events=size(1, 500),
                        precision=64, proposal=0, model=30, lcc=rng.choice((0, 0, 1)))
        n = size(1000, 200000)
        per = float(size(50, min(10000, n)))
        prop = rng.choice((0, 0, 1))
        model = 30 if prop else rng.choice((30, 30, 1))
        lcc = 0 if prop else rng.choice((0, 0, 1))
        return dict(kind=kind, cells=n, per_event=per, deltaf=rng.choice(("14mom", "rta")), quirk=rng.choice((0, 1)),
                    events=size(1, int(min(1000, 5.0e6 / per))), precision=rng.choice((32, 64)), proposal=prop,
                    model=model, lcc=lcc)
    if kind == "event":
        n = size(500, 60000)
        per = float(size(100, 5000))
        return dict(kind=kind, cells=n, per_event=per, deltaf=rng.choice(("ideal", "rta", "ce", "diffusion")),
                    eos=rng.choice((0, 9, 12, 14)), events=size(1, int(min(500, 1.0e6 / per))),
                    precision=rng.choice((32, 64)), decays=rng.choice((0, 1, 1)), model=rng.choice((30, 30, 1)),
                    lcc=rng.choice((0, 0, 1)))
    if kind == "batch":
        return dict(kind=kind, surfaces=rng.randint(2, 48), median=size(300, 6000), deltaf="14mom", quirk=0,
                    events=size(10, 150), precision=rng.choice((32, 32, 64)), proposal=rng.choice((0, 0, 1)))
    return dict(kind=kind, cells=size(1000, 20000), per_event=float(size(200, 1000)), deltaf="14mom", quirk=0,
                batch=64 * size(16, 128), steps=rng.randint(20, 100))


# ------------------------------------------------------------------ prepare
def train_network(ctx, per_event, seed, batch, steps):
    ctx.sample(max(1, int(5.0e5 / per_event)), seed=seed + 1)
    ctx.mlp_collect(2_000_000)
    ctx.mlp_init(1)
    ctx.mlp_train(batch=batch, steps=steps, lr=3e-3, seed=5)


def spectra_grid(case):
    """Species indices (pi+, K+, p first, then others), pT, phi and eta nodes
    with their weights: the reference's tables, or as many nodes of them."""
    sp, b = species(), bins()
    first = [int(np.nonzero(sp["pid"] == p)[0][0]) for p in (211, 321, 2212, -211, 3122)]
    idx = (first + [i for i in range(len(sp["pid"])) if i not in first])[:case["species"]]
    if case["mode"] == 0:
        step = (b["eta"].size - 1) // (case["eta"] - 1)
        eta, w = b["eta"][::step], b["eta_weight"][::step] * step
    else:
        eta, w = np.linspace(-2.5, 2.5, case["eta"]), None
    return dict(species=np.array(idx, dtype=np.int32), pT=b["pT"][:case["pT"]], phi=b["phi"][:case["phi"]], eta=eta,
                eta_weight=w)


def hadron_buffer(case):
    """The program's host buffer for the hadron list, with room for it."""
    count = per_event_of(case) * case["events"] * (case["surfaces"] if case["kind"] == "batch" else 1)
    room = (1.7 if case["kind"] == "event" else 1.25) * count * (1.9 if case.get("decays") else 1.0)
    return np.zeros(int(room + 20.0 * math.sqrt(room)) + 4096, dtype=iss_amd.HADRON_DTYPE)


def prepare(case, seed):
    kind = case["kind"]
    ctx = context(case)
    s = dict(case=case, ctx=ctx, seed=seed)
    if kind in ("sample", "event", "batch"):
        s["hadrons"] = hadron_buffer(case)
    if kind == "event":
        s["cells"] = lab_cells(case["cells"], case["per_event"], seed)
        s["eos"] = eos(case["eos"]) if case["eos"] else None
        if case["decays"]:
            ctx.set_decay_table(decays())
        return s
    if kind == "batch":
        n = batch_cells(case)
        cells = [lrf_cells({**case, "cells": int(k)}, seed * 1000 + i) for i, k in enumerate(n)]
        # 1 to 2 events - 1 of every surface, in no order
        s["events"] = (1 + np.arange(case["surfaces"]) * 7919 % (2 * case["events"] - 1)).astype(np.int32)
        ctx.set_surfaces_lrf(cells)
        if case["proposal"]:
            train_network(ctx, 0.05 * float(n.sum()), seed, 8192, 40)
        return s
    if case.get("boost_invariant"):
        ctx.set_surface_lab(binv_cells(case["cells"], seed))
    else:
        ctx.set_surface_lrf(lrf_cells(case, seed))
    if kind == "rows":
        # the first plain pass builds the Bessel tables; the caller's buffers
        ctx.compute_yields(precision=case["precision"])
        stride = ctx.row_stride(case["precision"])
        dt = torch.float64 if case["precision"] == 64 else torch.float32
        s["totals"] = torch.zeros(ctx.n_species, dtype=torch.float64, device="cuda")
        s["rows"] = torch.zeros((case["cells"], stride), dtype=dt, device="cuda")
    elif kind == "spectra":
        s["grid"] = spectra_grid(case)
    elif kind == "sample" and case["proposal"]:
        train_network(ctx, case["per_event"], seed, 8192, 40)
    elif kind == "train":
        ctx.sample(max(1, int(1.0e6 / case["per_event"])), seed=seed + 1)
        ctx.mlp_collect(10_000_000)
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------- run
def hadron_list(state):
    """The hadron list read back into the program's buffer, which it keeps
    from step to step: particle ids and the nine floats (slots past the list
    stay empty)."""
    ctx, buf = state["ctx"], state["hadrons"]
    rc = ctx.lib.iss_get_hadrons(ctx.h, buf.ctypes.data_as(ctypes.c_void_p), buf.size)
    if rc != 0:
        raise iss_amd.ISSError(f"hadron list: status {rc}")
    w = buf.view(np.int32).reshape(-1, 10)
    return {"pid": w[:, 0], "kinematics": w.view(np.float32)[:, 1:]}


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    mode = 1 if case.get("boost_invariant") else 2
    if kind == "yields":
        return {"totals": ctx.compute_yields(precision=case["precision"], hydro_mode=mode)}
    if kind == "rows":
        rows, tot = state["rows"], state["totals"]
        rc = ctx.compute_yields_noalloc(tot.data_ptr(), rows.data_ptr(), rows.numel(), precision=case["precision"])
        if rc != 0:
            raise iss_amd.ISSError(f"yields: status {rc}")
        return {"totals": tot, "rows": rows}
    if kind == "spectra":
        g = state["grid"]
        return {"dN": ctx.spectra(g["species"], g["pT"], g["phi"], g["eta"], g["eta_weight"], mode=case["mode"],
                                  precision=case["precision"])}
    if kind == "train":
        ctx.mlp_init(1)
        r = ctx.mlp_train(batch=case["batch"], steps=case["steps"], lr=3e-3, seed=state["seed"])
        return {"params": ctx.mlp_get_params(), "loss_first": r["loss_first"], "loss_last": r["loss_last"]}
    if kind == "batch":
        ctx.compute_yields(precision=case["precision"])
        ctx.sample_batch(state["events"], seed=state["seed"], precision=case["precision"], proposal=case["proposal"])
        seg, sizes = ctx.batch_layout()
        return {"segments": seg, "event_sizes": sizes, **hadron_list(state)}
    if kind == "event":
        ctx.set_surface_lab(state["cells"], state["eos"])
    out = {"yields": ctx.compute_yields(precision=case["precision"], hydro_mode=mode)}
    ctx.sample(case["events"], seed=state["seed"], hydro_mode=mode, y_LB=-1.0, y_RB=1.0, precision=case["precision"],
               proposal=case.get("proposal", 0), sampling_model=case["model"],
               local_charge_conservation=case["lcc"])
    if case.get("decays"):
        ctx.decay(seed=state["seed"] + 17)
    out["counts"] = ctx.event_counts()
    out.update(hadron_list(state))
    return out


# --------------------------------------------------------------------- work
def per_event_of(case):
    if case.get("boost_invariant"):
        return 1090.0   # two units of rapidity of the 180 fm^2 surface
    if case["kind"] == "batch":
        return 0.05 * float(np.mean(batch_cells(case)))
    return case.get("per_event", 0.05 * case["cells"])


def work(case):
    """Bytes: cells read once (six floats for the yields, the record for the
    rest), outputs written once.  Operations: 20 per yield of one series term,
    40 per spectrum integrand, 450 per hadron (two trials), the network's
    three products forward and twice that backward."""
    kind, n, ns = case["kind"], case.get("cells", 0), len(species()["pid"])
    esz = 8 if case.get("precision") == 64 else 4
    if kind == "yields":
        return {"bytes": 24.0 * n + 8.0 * ns, "flops": 25.0 * n * ns}
    if kind == "rows":
        return {"bytes": 24.0 * n + float(esz) * n * ns + 8.0 * ns, "flops": 25.0 * n * ns}
    if kind == "spectra":
        points = case["species"] * case["pT"] * case["phi"] * case["eta"]
        out = points // case["eta"] if case["mode"] == 0 else points
        return {"bytes": 112.0 * n + 8.0 * out, "flops": 40.0 * n * points}
    if kind == "train":
        macs = 14 * 64 + 64 * 64 + 64 * 8
        return {"bytes": 6.0 * case["batch"] * case["steps"] + 4.0 * macs, "flops": 6.0 * macs * case["batch"] * case["steps"]}
    hadrons = per_event_of(case) * case["events"] * (case["surfaces"] if kind == "batch" else 1)
    cells = int(batch_cells(case).sum()) if kind == "batch" else n
    final = 1.9 * hadrons if case.get("decays") else hadrons
    return {"bytes": (136.0 if kind == "event" else 112.0) * cells + 40.0 * final, "flops": 25.0 * cells * ns + 450.0 * hadrons}


# -------------------------------------------------------------------- exact
def bessel_table():
    """K_1, K_2, K_3 on x = 0.5 + 0.05 i: the yields interpolate linearly in
    this table, which is part of their definition."""
    x = 0.5 + 0.05 * torch.arange(7991, dtype=torch.float64, device="cuda")
    k0, k1 = torch.special.modified_bessel_k0(x), torch.special.modified_bessel_k1(x)
    k2 = k0 + 2.0 / x * k1
    return {1: k1, 2: k2, 3: k1 + 4.0 / x * k2}


def interpolate(table, arg):
    t = (arg - 0.5) / 0.05
    i = t.to(torch.int64)
    f = t - i
    return (1.0 - f) * table[i] + f * table[i + 1]


def bulk_14mom(T, muB):
    """The 14-moment coefficients, bilinear in (T, mu_B)."""
    k = kind11()
    ft, fm = (T - k["T0"]) / k["dT"], (muB - k["mu0"]) / k["dmu"]
    it, im = ft.to(torch.int64), fm.to(torch.int64)
    x, y = ft - it, fm - im
    t1, t2 = it.clamp(0, k["nT"] - 1), (it + 1).clamp(0, k["nT"] - 1)
    m1, m2 = im.clamp(0, k["nmu"] - 1), (im + 1).clamp(0, k["nmu"] - 1)
    v = []
    for name in ("c0", "c1", "c2"):
        g = torch.tensor(np.asarray(k[name]).reshape(k["nT"], k["nmu"]), dtype=torch.float64, device="cuda")
        v.append(g[t1, m1] * (1 - x) * (1 - y) + g[t1, m2] * (1 - x) * y + g[t2, m2] * x * y + g[t2, m1] * x * (1 - y))
    return (v[0] - v[2]) / T ** 4, v[1] / T ** 3, (4 * v[2] - v[0]) / T ** 4


def device_cells(case, seed):
    return torch.tensor(lrf_cells(case, seed), device="cuda").double()


def exact_rows(case, seed):
    sp = species()
    if case.get("boost_invariant"):
        lab = torch.tensor(binv_cells(case["cells"], seed), device="cuda").double()
        T, muB, Pi = lab[:, 13], lab[:, 16], torch.zeros_like(lab[:, 13])
        # u.dsigma of a cell with dsigma along tau only, as the float record holds it
        u0 = torch.sqrt(1 + lab[:, 9] ** 2 + lab[:, 10] ** 2)
        dsu = (lab[:, 0] * lab[:, 4] * u0).float().double()
    else:
        c = device_cells(case, seed)
        T, muB, dsu, Pi = c[:, 13], c[:, 16], c[:, 4], c[:, 19]
    K = bessel_table()
    bulk = bulk_14mom(T, muB) if case["deltaf"] == "14mom" else None
    cols = []
    for m, g, B, sg in zip(sp["mass"], sp["g"], sp["B"], sp["sign"]):
        m, g, B, sg = float(m), float(g), float(B), float(sg)
        lam = torch.exp(B * muB / T)
        r = [torch.zeros_like(T) for _ in range(4)]
        for n in range(1, (10 if m < 0.7 else 1) + 1):
            k2 = interpolate(K[2], n * m / T)
            w = (-sg) ** (n - 1) * lam ** n
            r[0] += w / n * k2
            if bulk:
                k1, k3 = interpolate(K[1], n * m / T), interpolate(K[3], n * m / T)
                r[1] += w * k2
                r[2] += w * (m / T * k1 + 3 * k2 / n)
                r[3] += w * (m / T * k2 + 3 * k3 / n)
        v = m * m * T * r[0]
        if bulk:
            v = v + Pi * (m ** 4 * T * r[1] * bulk[0] + m * m * T * T * r[2] * B * bulk[1] + m ** 3 * T * T * r[3] * bulk[2])
        cols.append((g / (2 * math.pi ** 2 * HBARC ** 3) * dsu * v).clamp_min(0.0))
    return cols


def exact_spectra(case, seed):
    sp, g = species(), spectra_grid(case)
    cells = device_cells(case, seed)
    d = dict(dtype=torch.float64, device="cuda")
    pT, phi, eta = (torch.tensor(np.asarray(g[k]), **d) for k in ("pT", "phi", "eta"))
    cph, sph = torch.cos(phi), torch.sin(phi)
    mode0 = case["mode"] == 0
    w = torch.tensor(np.asarray(g["eta_weight"]), **d) if mode0 else None
    nodes = eta.numel()
    out = torch.zeros((len(g["species"]), nodes if not mode0 else 1, pT.numel(), phi.numel()), **d)
    step = max(1, int(2.5e8 // (nodes * pT.numel() * phi.numel())))
    for c0 in range(0, cells.shape[0], step):
        c = cells[c0:c0 + step]
        shape = lambda v: v.reshape(-1, 1, 1, 1)  # noqa: E731
        T, muB, Pi = c[:, 13], c[:, 16], c[:, 19]
        u = [c[:, 8 + k] for k in range(4)]
        ds = [c[:, 4 + k] for k in range(4)]
        y = c[:, 3:4] - eta[None] if mode0 else eta[None].expand(c.shape[0], -1)
        bulk = bulk_14mom(T, muB) if case["deltaf"] == "14mom" else None
        xx, xy, xz, yy, yz = (c[:, 20 + k] for k in range(5))
        ipi = 1.0 / (2 * T * T * (c[:, 12] + c[:, 14]))
        ch, sh = torch.cosh(y), torch.sinh(y)
        for i, s in enumerate(g["species"]):
            m, gs, B, sg = float(sp["mass"][s]), float(sp["g"][s]), float(sp["B"][s]), float(sp["sign"][s])
            mT = torch.sqrt(pT * pT + m * m)
            # rest-frame components, linear in the lab momentum: mT times a
            # (cell, node) factor plus a (cell, pT, phi) term
            px, py = pT[:, None] * cph[None], pT[:, None] * sph[None]
            iu = 1.0 / (u[0] + 1.0)
            pu = shape(u[1])[..., 0] * px[None] + shape(u[2])[..., 0] * py[None]
            a0 = u[0][:, None] * ch - u[3][:, None] * sh
            gk = u[3][:, None] * sh * iu[:, None] - ch
            a = [u[1][:, None] * gk, u[2][:, None] * gk, sh + u[3][:, None] * gk]
            P = [px[None] + pu * shape(iu * u[1])[..., 0], py[None] + pu * shape(iu * u[2])[..., 0],
                 pu * shape(iu * u[3])[..., 0]]
            M = mT[None, None, :, None]
            full = lambda ak, Pk: ak[:, :, None, None] * M + Pk[:, None]  # noqa: E731
            E = full(a0, -pu)
            l = [full(a[k], P[k]) for k in range(3)]
            f0 = (E - shape(B * muB)).mul_(shape(1.0 / T)).exp_().add_(sg).reciprocal_()
            pds = E * shape(ds[0])
            for k in range(3):
                pds.addcmul_(l[k], shape(ds[1 + k]).expand_as(E))
            if bulk:
                W = (l[0] * shape(xx) + l[1] * shape(2 * xy) + l[2] * shape(2 * xz)).mul_(l[0])
                W += (l[1] * shape(yy) + l[2] * shape(2 * yz)).mul_(l[1])
                W -= (l[2] * l[2]).mul_(shape(xx + yy))
                W.mul_(shape(ipi))
                W += (E * shape(bulk[2]) + shape(B * bulk[1])).mul_(E).mul_(shape(Pi)).add_(shape(Pi * bulk[0] * m * m))
                W.mul_(1.0 - sg * f0)
                pds.mul_(W.clamp_(-1.0, 1.0).add_(1.0))
            pds.mul_(f0)
            pre = gs / (8 * math.pi ** 3) / HBARC ** 3
            if mode0:
                out[i, 0] += pre * torch.einsum("k,kij->ij", w, pds.sum(0))
            else:
                out[i] += pre * pds.sum(0)
    return (out[:, 0] if mode0 else out).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "spectra":
        return {"dN": exact_spectra(case, seed)}
    if kind not in ("yields", "rows"):
        return None     # random draws: no value of their own
    cols = exact_rows(case, seed)
    totals = torch.stack([c.sum() for c in cols])
    if kind == "yields":
        return {"totals": totals.cpu().numpy()}
    rows = torch.zeros((case["cells"], (len(cols) + 15) // 16 * 16 if case["precision"] == 32 else (len(cols) + 7) // 8 * 8),
                       dtype=torch.float64, device="cuda")
    for s, col in enumerate(cols):
        rows[:, s] = col
    return {"totals": totals, "rows": rows}
