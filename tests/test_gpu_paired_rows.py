"""Lists with enough bonds for the two directions of a bond to share one row of radial functions (k_edge_pairs): symmetric
lists, lists in which one direction of a bond is missing, lists that hold bonds twice, bond vectors that were rounded
differently in the two directions, atoms with more than 80 neighbours, chunks that cut bonds, chunks of isolated atoms, against
the oracle on the same list."""
import numpy as np
import pytest

import cases
from grace_runtime_amd import kk, synth
from oracle import grace_oracle as g1
from oracle import grace_oracle_2l as g2

pytestmark = pytest.mark.gpu


def _list(variant):
    """types, offset, j, rij of a two-element bcc cell"""
    # "long": about 100 neighbours inside the cutoff of 5 A, more than the 80 that one step of the search takes
    pos, cell = synth.bcc_supercell(2.2, 7) if variant == "long" else synth.bcc_supercell(3.165, 8)
    pos = synth.jitter(pos, 0.08, 4)
    rng = np.random.default_rng(9)
    types = rng.integers(1, 3, len(pos)).astype(np.int32)
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True] * 3, 5.4)
    rij = cases.bond_vectors(pos, perm, offset, j, image, shifts)
    i = np.repeat(np.arange(len(pos)), np.diff(offset))
    if variant == "holes":
        keep = rng.random(len(j)) > 0.15
        i, j, rij = i[keep], j[keep], rij[keep]
    if variant == "twice":
        order = np.sort(np.concatenate([np.arange(len(j)), rng.choice(len(j), len(j) // 8, replace=False)]))
        i, j, rij = i[order], j[order], rij[order]
    if variant == "rounded":
        rij = rij * (1.0 + 2e-16 * rng.integers(-2, 3, rij.shape))
    types = types[perm]
    if variant == "gas":    # 700 atoms without a neighbour: chunks of 300 atoms that hold no bond, between others and at the end
        late = i >= 512
        i, j = i + 700 * late, j + 700 * (j >= 512)
        types = np.concatenate([types[:512], rng.integers(1, 3, 700).astype(np.int32), types[512:], np.ones(700, np.int32)])
    offset = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=len(types)))]).astype(np.int64)
    assert len(j) > 32768
    return types, offset, j.astype(np.int32), rij


_oracle = {}


@pytest.mark.parametrize("precision,chunk", [(64, 0), (32, 0), (64, 300)])
@pytest.mark.parametrize("variant", ["plain", "holes", "twice", "rounded", "long", "gas"])
@pytest.mark.parametrize("model", ["mix2", "l2mix"])
def test_shared_rows_equal_the_oracle(model_dir, model, variant, precision, chunk):
    path = cases.model_file(model_dir, model)
    types, offset, j, rij = _list(variant)
    eng = kk.Engine(kk.Model(path), ["Mo", "W"], precision)
    eng.set_chunksize(chunk)
    out = eng.compute(types, offset, j, rij=rij, energies=True)
    if (model, variant) not in _oracle:
        _oracle[(model, variant)] = g1.compute_1l(g1.Model1L(path), types - 1, offset, j, rij) if model == "mix2" else \
            g2.compute_2l(g2.Model2L(path), types - 1, offset, j, rij)
    # the bounds of the other parity tests: 1e-10 eV/atom, 1e-9 eV/A in fp64, the fp32 gate of the reference else
    tol = (1e-10, 1e-9, 1e-10, 1e-9) if precision == 64 else (1e-6, 2e-5, 1e-5, 1e-5)
    cases.check_against(out, _oracle[(model, variant)], len(types), *tol)
