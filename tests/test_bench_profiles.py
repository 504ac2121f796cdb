"""The profile entries that the benchmark line quotes: the kernel's own
instance, not the first one of its name."""
import json
import os

import pytest

import bench


@pytest.fixture
def profiles(tmp_path, monkeypatch):
    os.mkdir(tmp_path / "profiles")
    rows = {"k_yield_rows<double, 11, false>": 2, "k_yield_rows<float, 0, false>": 1, "k_yield_rows<float, 11, false>": 4,
            "k_setup<false>": 3, "k_setup<true>": 5, "k_trials": 7}
    u = {"N_SIMD": 1024, **{k: {"dispatches": n, "name": k} for k, n in rows.items()}}
    for f in ("utilisation.json", "traffic.json"):
        (tmp_path / "profiles" / f).write_text(json.dumps(u))
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))


@pytest.mark.parametrize("kernel,precision,want", [
    ("k_yield_rows", 32, "k_yield_rows<float, 11, false>"), ("k_yield_rows", 64, "k_yield_rows<double, 11, false>"),
    ("k_yield_rows", 0, "k_yield_rows<float, 11, false>"), ("k_setup", 0, "k_setup<true>"), ("k_trials", 0, "k_trials"),
    ("k_trials", 32, "k_trials"), ("k_absent", 0, None)])
def test_entry_is_the_kernels_own(profiles, kernel, precision, want):
    for f in (bench.hw_from_profiles, bench.traffic_from_profiles):
        e = f(kernel, precision)
        assert (e and e["name"]) == want


def test_without_profiles(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.hw_from_profiles("k_trials") is None and bench.traffic_from_profiles("k_trials") is None
