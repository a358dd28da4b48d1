"""The A basis and the bond reverse over atoms whose bonds end around the tiles of 16 and the rounds of 32 and 64 that their kernels
take at once: clusters in which every atom sees all others (n - 1 bonds each), against the oracle; with radial tables evaluated in
the kernels against the same tables as rows (GRACE_HIP_TABLE_ROWS; bond_force, atom_scatter: libgrace/include/grace/fused_cpu.h:
836-860,1027-1050; tables: libgrace/src/fused_1l.cpp:102-129)."""
import numpy as np
import pytest

import cases
from grace_runtime_amd import kk

pytestmark = pytest.mark.gpu

SIZES = [2, 16, 17, 18, 32, 33, 34, 49, 64, 65, 66, 97]


def cluster(n, radius):
    """n points in a ball, none closer than a bit over half the mean distance"""
    rng = np.random.default_rng(n)
    out, gap = [], 0.55 * radius * (4.0 / n) ** (1.0 / 3.0)
    while len(out) < n:
        p = rng.uniform(-radius, radius, 3)
        if np.linalg.norm(p) < radius and all(np.linalg.norm(p - q) > gap for q in out):
            out.append(p)
    return np.array(out)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model,species,cutoff", [("config1", ["W"], 6.0), ("mix2", ["Mo", "W"], 5.0)])
@pytest.mark.parametrize("n", SIZES)
def test_bonds_around_the_tile_sizes(model_dir, monkeypatch, n, model, species, cutoff, precision):
    path = cases.model_file(model_dir, model)
    pos = cluster(n, 0.49 * cutoff)
    types = (np.arange(n) % len(species) + 1).astype(np.int32)
    cell, pbc = 30.0 * np.eye(3), [False, False, False]
    m = kk.Model(path)
    out = kk.System(m, species, skin=0.0, precision=precision).compute(types, pos, cell, pbc)
    ref = cases.oracle_reference(model_dir, model, pos, cell, pbc, types)
    fs = max(1.0, np.abs(ref["forces"]).max())
    tol = 1e-10 if precision == 64 else 2e-6
    assert abs(out["energy"] - ref["energy"]) / n < tol * fs
    assert np.abs(out["forces"] - ref["forces"]).max() < 10 * tol * fs
    assert np.abs(out["virial"] - ref["virial"]).max() < 100 * tol * fs
    inside = kk.System(m, species, skin=0.0, precision=precision, spline=200).compute(types, pos, cell, pbc)
    monkeypatch.setenv("GRACE_HIP_TABLE_ROWS", "1")
    rows = kk.System(m, species, skin=0.0, precision=precision, spline=200).compute(types, pos, cell, pbc)
    assert abs(inside["energy"] - rows["energy"]) / n < tol * fs
    assert np.abs(inside["forces"] - rows["forces"]).max() < 10 * tol * fs


@pytest.mark.parametrize("tables", [0, 200])
@pytest.mark.parametrize("model,species,cutoff", [("config1", ["W"], 6.0), ("mix2", ["Mo", "W"], 5.0)])
@pytest.mark.parametrize("n", SIZES)
def test_many_atoms_with_bonds_around_the_tile_sizes(model_dir, n, model, species, cutoff, tables):
    """fp32, where the bond reverse takes one tile at a time up to two atoms per CU and two beyond: a cluster among as many copies as
    make more atoms than that, against the cluster by itself; forces, which the two forms give in the same terms, and the virial"""
    m = kk.Model(cases.model_file(model_dir, model))
    pos = cluster(n, 0.49 * cutoff)
    types = (np.arange(n) % len(species) + 1).astype(np.int32)
    copies = 520 // n + 1
    side = int(np.ceil(copies ** (1.0 / 3.0)))
    at = np.stack(np.unravel_index(np.arange(copies), (side,) * 3), -1) * 3.0 * cutoff
    many = (pos[None] + at[:, None]).reshape(-1, 3)
    pbc = [False, False, False]
    one = kk.System(m, species, skin=0.0, precision=32, spline=tables).compute(types, pos, 30.0 * np.eye(3), pbc)
    out = kk.System(m, species, skin=0.0, precision=32, spline=tables).compute(np.tile(types, copies), many, 200.0 * np.eye(3), pbc)
    fs = max(1.0, np.abs(one["forces"]).max())
    tol = 2e-6
    assert np.abs(out["forces"].reshape(copies, n, 3) - one["forces"]).max() < 10 * tol * fs
    assert np.abs(out["virial"] - copies * one["virial"]).max() < 100 * tol * fs * copies
