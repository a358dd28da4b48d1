"""Atoms whose numbers of bonds lie around the tiles of 16 and the rounds of 64 bonds of k_scatter_a_mfma, k_scatter_a_tab and
k_bond_bwd, with rows and with radial tables, against the fp64 oracle at the bounds of the other parity tests."""
import numpy as np
import pytest

import cases
from grace_runtime_amd import kk
from oracle import grace_oracle as g1

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("intervals", [0, 1024])
@pytest.mark.parametrize("model", ["mix2", "cut2"])
def test_bond_counts(model_dir, model, intervals, precision):
    path = cases.model_file(model_dir, model)
    species = {"mix2": ["Mo", "W"], "cut2": ["Al", "Ni"]}[model]
    om = g1.Model1L(path)
    om.spline = intervals
    engine = kk.Engine(kk.Model(path), species, precision)
    engine.set_spline(intervals)
    rng = np.random.default_rng(7)
    counts = np.array([0, 1, 15, 16, 17, 48, 63, 64, 65, 79, 80, 81, 127, 128, 129, 192, 200, 0])
    n = len(counts)
    offset = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    j = rng.integers(0, n, offset[-1]).astype(np.int32)
    d = rng.normal(size=(offset[-1], 3))
    shortest = float(engine.cutoff_matrix().min())
    rij = d / np.linalg.norm(d, axis=1)[:, None] * rng.uniform(0.4 * shortest, 0.95 * shortest, (offset[-1], 1))
    types = rng.integers(1, 3, n).astype(np.int32)
    ref = g1.compute_1l(om, types - 1, offset, j, rij)
    out = engine.compute(types, offset, j, rij, energies=True)
    fs = max(1.0, np.abs(ref["forces"]).max())
    tol = 1e-10 if precision == 64 else 2e-6
    assert abs(out["energy"] - ref["energy"]) / n < tol * fs
    assert np.abs(out["energies"] - ref["energies"]).max() < tol * fs
    assert np.abs(out["forces"] - ref["forces"]).max() < 10 * tol * fs
    assert np.abs(out["virial"] - ref["virial"]).max() < 100 * tol * fs
