"""The job GEMMs of GRACE-3L over few and many tiles of atoms (k_gemm_few, k_gemm_wide) and the contractions joined in one
launch: structures whose atoms fill one tile, part of a tile and a tile and one atom, and batches whose tiles pass the
sizes where the launch changes its kernel, against the oracle.  Widths of 32 and 64 channels, joined and single launches
(l3pad, l3el: other widths, weights per element)."""
import numpy as np
import pytest

import cases
from grace_runtime_amd import kk
from oracle import grace_oracle_3l as g3

pytestmark = pytest.mark.gpu

_oracle = {}


def _structure(natoms, species):
    pos, cell, pbc, types = cases.structure_config4(natoms=natoms, seed=natoms)
    return pos, cell, pbc, (types % species + 1).astype(np.int32)


def _reference(model, path, names, natoms, species):
    if (model, natoms) not in _oracle:
        pos, cell, pbc, types = _structure(natoms, species)
        rc = float(kk.Engine(kk.Model(path), names, 64).cutoff_matrix().max())
        perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, pbc, rc)
        ref = g3.compute_3l(g3.Model3L(path), kk.Model(path).type2mu(names)[1:][types[perm] - 1], offset, j,
                            cases.bond_vectors(pos, perm, offset, j, image, shifts))
        f = np.zeros((natoms, 3))
        f[perm] = ref["forces"]
        _oracle[(model, natoms)] = (ref["energy"], f)
    return _oracle[(model, natoms)]


# copies of a cell: with the 36 .. 72 jobs of these models the launches change their kernel between 2 and 8 groups of 8 tiles
@pytest.mark.parametrize("model,natoms,copies,precision", [
    ("config4", 1, 1, 64), ("config4", 15, 1, 64), ("config4", 17, 1, 64), ("config4", 17, 40, 64), ("config4", 17, 40, 32),
    ("config4", 17, 130, 64), ("l3pad", 17, 3, 64), ("l3el", 17, 3, 64), ("l3mix", 33, 20, 64)])
def test_few_and_many_tiles(model_dir, model, natoms, copies, precision):
    path = cases.model_file(model_dir, model)
    m = kk.Model(path)
    names = list(m.element_names)[:2] if model != "config4" else ["Mo", "W"]
    pos, cell, pbc, types = _structure(natoms, len(names))
    energy, forces = _reference(model, path, names, natoms, len(names))
    b = kk.Batch(m, names, precision=precision)
    out = b.compute([natoms] * copies, np.tile(types, copies), np.tile(pos, (copies, 1)), np.tile(cell, (copies, 1, 1)), np.tile(pbc, (copies, 1)))
    # the bounds of the other parity tests: 1e-10 eV/atom and 1e-9 eV/A in fp64, the fp32 gate of the reference else
    te, tf = (1e-10, 1e-9) if precision == 64 else (1e-6, 2e-5)
    fs = max(1.0, np.abs(forces).max())
    assert np.abs(out["energy"] - energy).max() < te * natoms * fs
    assert np.abs(out["forces"].reshape(copies, natoms, 3) - forces).max() < tf * fs
