"""The element-dependent reduces (k_reduce_fwd, k_reduce_sum, k_reduce_bwd) where their launches can go wrong: a function of the
chain that several functions of I1 and rho collect at once (more than two feeds of one adjoint row take a second launch that
adds), a layer of more reduces than one launch takes, tiles that are whole, part or one atom over, and structures and batches on
both sides of the number of tiles from which a reduce is no longer split over several blocks.  Against the fp64 oracle at the bounds of the other parity tests."""
import os

import numpy as np
import pytest

import cases
from grace_runtime_amd import kk
from oracle import grace_oracle_2l as g2

pytestmark = pytest.mark.gpu
TOL = {64: (1e-10, 1e-9), 32: (1e-6, 2e-5)}    # energy per atom, forces


def _base(model_dir, model):
    return os.path.join(cases.REF_FIXTURES, model + ".npz") if model == "grace_2l_small" else cases.model_file(model_dir, model)


def _shared_model(base, tmp_path, extra):
    """the model with the first collected function of every source of I1 connected to `extra` more functions of I1"""
    d = dict(np.load(base, allow_pickle=False))
    nf = 1 + max(int(d[k].max()) for k in d if k.startswith("I1_total_sum_ind_"))
    assert nf > extra
    for k in [k for k in d if k.startswith("I1_total_sum_ind_")]:
        src = k[len("I1_total_sum_ind_"):]
        first = int(d[k].ravel()[0])
        for key, values in (("I1_collect_ind_", [int(d["I1_collect_ind_" + src].ravel()[0])] * extra), ("I1_w_l_tile_", [int(d["I1_w_l_tile_" + src].ravel()[0])] * extra),
                            ("I1_total_sum_ind_", [(first + q) % nf for q in range(1, extra + 1)])):
            old = d[key + src]
            d[key + src] = np.concatenate([old, np.array(values, old.dtype).reshape((extra,) + old.shape[1:])])
    path = os.path.join(str(tmp_path), "shared.npz")
    np.savez(path, **d)
    return path


def _oracle(path, pos, cell, types, species):
    model = kk.Model(path)
    rc = float(kk.Engine(model, species, 64).cutoff_matrix().max())
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True] * 3, rc)
    ref = g2.compute_2l(g2.Model2L(path), model.type2mu(species)[1:][types[perm] - 1], offset, j, cases.bond_vectors(pos, perm, offset, j, image, shifts))
    f = np.zeros((len(pos), 3))
    f[perm] = ref["forces"]
    return ref["energy"], f


# grace_2l_small: 16 channels, the chain stage by stage; config5: 32 channels, the generated chain, whose adjoint rows are written
@pytest.mark.parametrize("model,extra,precision", [("grace_2l_small", 1, 64), ("grace_2l_small", 3, 64), ("config5", 1, 64), ("config5", 3, 64), ("config5", 3, 32)])
def test_one_function_collected_several_times(model_dir, tmp_path, model, extra, precision):
    path = _shared_model(_base(model_dir, model), tmp_path, extra)
    species = [str(n) for n in kk.Model(path).element_names][:2]
    rng = np.random.default_rng(3)
    pos = np.array([[x, y, z] for x in range(3) for y in range(3) for z in range(2)]) * 2.6 + rng.normal(0, 0.1, (18, 3))
    cell, types = np.diag([7.8, 7.8, 5.2]), rng.integers(1, 3, 18).astype(np.int32)
    energy, forces = _oracle(path, pos, cell, types, species)
    out = kk.System(kk.Model(path), species, 0.5, precision=precision).compute(types, pos, cell, np.array([True] * 3))
    fs, (te, tf) = max(1.0, np.abs(forces).max()), TOL[precision]
    assert abs(out["energy"] - energy) < te * len(pos) * fs
    assert np.abs(out["forces"] - forces).max() < tf * fs


def _many_functions_model(base, tmp_path):
    """the model with four more functions of I1, from A and AA alone, which feed I beside the first four: nine reduces of layer 1
    where a launch takes eight"""
    d = dict(np.load(base, allow_pickle=False))
    nf = int(d["I1_n_funcs"][0])
    assert nf == 4
    d["I1_n_funcs"] = d["I1_n_funcs"] * 2
    for src in ("I1_{}_A", "I1_{}_AA", "I_{}_I1"):
        for key, plus in (("collect_ind", nf if src.startswith("I_") else 0), ("w_l_tile", 0), ("total_sum_ind", 0 if src.startswith("I_") else nf)):
            old = d[src.format(key)]
            d[src.format(key)] = np.concatenate([old, old + plus])
    path = os.path.join(str(tmp_path), "functions.npz")
    np.savez(path, **d)
    return path


# copies of a cell of two or more tiles (two species: every cell's tiles hold both).  With 256 CUs the five reduces of layer 1 go to
# 512 / (5 x tiles) blocks each, no more than an eighth of their functions: one tile, three blocks up to 34 tiles, two up to 51, one
# beyond; the single reduce of layer 2 is whole from 257 tiles on.  With nine reduces the eight of the first launch are whole from
# 33 tiles on, the ninth is in parts.  Tiles of these batches: 17 atoms x copies / 16 and up to one more
@pytest.mark.parametrize("model,natoms,copies,precision", [
    ("grace_2l_small", 2, 1, 64), ("config5", 2, 1, 64), ("config5", 15, 1, 64), ("config5", 17, 1, 32), ("grace_2l_small", 17, 2, 64), ("config5", 17, 31, 64),
    ("config5", 17, 40, 64), ("config5", 17, 40, 32), ("grace_2l_small", 17, 40, 64), ("config5", 17, 50, 64), ("grace_2l_small", 17, 150, 64),
    ("config5", 17, 150, 64), ("config5", 17, 150, 32), ("config5", 17, 245, 64), ("functions", 17, 1, 64), ("functions", 17, 20, 32), ("functions", 17, 40, 64)])
def test_few_and_many_tiles(model_dir, tmp_path, model, natoms, copies, precision):
    path = _many_functions_model(_base(model_dir, "config5"), tmp_path) if model == "functions" else _base(model_dir, model)
    species = [str(n) for n in kk.Model(path).element_names][:2]
    rng = np.random.default_rng(natoms)
    grid = np.array([[x, y, z] for x in range(3) for y in range(3) for z in range(2)])[:natoms]
    pos = grid * 2.6 + rng.normal(0, 0.1, (natoms, 3))
    cell, types = np.diag([7.8, 7.8, 5.2]), rng.integers(1, 3, natoms).astype(np.int32)
    energy, forces = _oracle(path, pos, cell, types, species)
    out = kk.Batch(kk.Model(path), species, precision=precision).compute([natoms] * copies, np.tile(types, copies), np.tile(pos, (copies, 1)),
                                                                         np.tile(cell, (copies, 1, 1)), np.ones((copies, 3), bool))
    fs, (te, tf) = max(1.0, np.abs(forces).max()), TOL[precision]
    assert np.abs(out["energy"] - energy).max() < te * natoms * fs
    assert np.abs(out["forces"].reshape(copies, natoms, 3) - forces).max() < tf * fs
