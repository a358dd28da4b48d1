"""The readout kernels (k_energy_hidden, k_energy_2l_hidden and the general k_energy, k_energy_2l) over the shapes of the network
on both sides of the rule that chooses between them, with both activations and the legacy layer norm, and with atom counts
around the 16 of a block and above the blocks of a launch.  Against the fp64 oracle at the bounds of the other parity tests; a
large periodic cell against the small one that it repeats."""
import os

import numpy as np
import pytest

import cases
from grace_runtime_amd import kk
from oracle import grace_oracle as g1
from oracle import grace_oracle_2l as g2

pytestmark = pytest.mark.gpu
ORACLE = {"config1": (g1.Model1L, g1.compute_1l), "config5": (g2.Model2L, g2.compute_2l)}


def _with_readout(model_dir, tmp_path, model, widths, act, scale):
    """the model with a readout network of these hidden widths"""
    d = dict(np.load(cases.model_file(model_dir, model), allow_pickle=False))
    rng = np.random.default_rng(sum(widths) + act)
    dims = [d["energy_mlp_W0"].shape[0], *widths, 1]
    for k in range(len(dims) - 1):
        d[f"energy_mlp_W{k}"] = rng.normal(0, 1, (dims[k], dims[k + 1]))
        d[f"energy_mlp_norm{k}"] = np.float64(1.0 / np.sqrt(dims[k]))
    d["energy_mlp_n_layers"], d["energy_mlp_activation"] = np.int64(len(dims) - 1), np.int64(act)
    if scale:
        d["energy_mlp_scale"] = rng.uniform(0.5, 1.5, dims[0])
    path = os.path.join(str(tmp_path), "readout.npz")
    np.savez(path, **d)
    return path


def _cell(natoms, species):
    rng = np.random.default_rng(natoms)
    grid = np.array([[x, y, z] for x in range(3) for y in range(3) for z in range(2)])[:natoms]
    return grid * 2.6 + rng.normal(0, 0.1, (natoms, 3)), np.diag([7.8, 7.8, 5.2]), rng.integers(1, species + 1, natoms).astype(np.int32)


def _check(path, model, species, natoms):
    make, compute = ORACLE[model]
    pos, cell, types = _cell(natoms, len(species))
    m = kk.Model(path)
    rc = float(kk.Engine(m, species, 64).cutoff_matrix().max())
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True] * 3, rc)
    ref = compute(make(path), m.type2mu(species)[1:][types[perm] - 1], offset, j, cases.bond_vectors(pos, perm, offset, j, image, shifts))
    out = kk.System(m, species, 0.5).compute(types, pos, cell, np.array([True] * 3), energies=True)
    fs = max(1.0, np.abs(ref["forces"]).max())
    assert abs(out["energy"] - ref["energy"]) < 1e-10 * natoms * fs
    assert np.abs(out["energies"][perm] - ref["energies"]).max() < 1e-10 * fs
    assert np.abs(out["forces"][perm] - ref["forces"]).max() < 1e-9 * fs


# 240 hidden units are the most whose weights a block stages; wider and deeper networks run the general kernels
@pytest.mark.parametrize("model", ["config1", "config5"])
@pytest.mark.parametrize("widths,act,scale", [((1,), 0, False), ((15,), 1, False), ((17,), 0, True), ((64,), 1, True), ((240,), 0, False), ((241,), 0, False),
                                              ((20, 12), 1, False)])
def test_networks(model_dir, tmp_path, model, widths, act, scale):
    path = _with_readout(model_dir, tmp_path, model, widths, act, scale)
    _check(path, model, [str(n) for n in kk.Model(path).element_names][:2], 17)


@pytest.mark.parametrize("model", ["config1", "config5"])
@pytest.mark.parametrize("natoms", [1, 15, 16, 18])
def test_atom_counts(model_dir, model, natoms):
    path = cases.model_file(model_dir, model)
    _check(path, model, [str(n) for n in kk.Model(path).element_names][:2], natoms)


# more atoms than the 1024 blocks of a launch hold: as one structure, and as a batch with its own record per structure
@pytest.mark.parametrize("model", ["config1", "config5"])
def test_more_atoms_than_blocks(model_dir, model):
    path = cases.model_file(model_dir, model)
    species = [str(n) for n in kk.Model(path).element_names][:2]
    pos, cell, types = _cell(18, len(species))
    reps = np.array([[x, y, z] for x in range(10) for y in range(10) for z in range(10)])
    pbc = np.array([True] * 3)
    one = kk.System(kk.Model(path), species, 0.5).compute(types, pos, cell, pbc)
    fs = max(1.0, np.abs(one["forces"]).max())
    big = kk.System(kk.Model(path), species, 0.5).compute(np.tile(types, 1000), (pos[None] + (reps @ cell)[:, None]).reshape(-1, 3), 10 * cell, pbc)
    assert abs(big["energy"] - 1000 * one["energy"]) < 1e-10 * 18000 * fs
    assert np.abs(big["forces"].reshape(1000, 18, 3) - one["forces"]).max() < 1e-9 * fs
    many = kk.Batch(kk.Model(path), species).compute([18] * 1000, np.tile(types, 1000), np.tile(pos, (1000, 1)), np.tile(cell, (1000, 1, 1)),
                                                     np.ones((1000, 3), bool))
    assert np.abs(many["energy"] - one["energy"]).max() < 1e-10 * 18 * fs
    assert np.abs(many["forces"].reshape(1000, 18, 3) - one["forces"]).max() < 1e-9 * fs
