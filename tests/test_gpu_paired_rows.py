"""Lists with enough bonds for the two directions of a bond to share one row of radial functions (k_edge_pairs): symmetric
lists, lists in which one direction of a bond is missing, lists that hold bonds twice, bond vectors that were rounded
differently in the two directions or differ by more than that, atoms with more than 80 neighbours, chunks that cut bonds, chunks of isolated atoms, against
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
    if variant == "apart":    # the directions of a bond differ by 1e-6 of its length: no row stands for both
        rij = rij * (1.0 + 1e-6 * (i > j))[:, None]
    types = types[perm]
    if variant == "gas":    # 700 atoms without a neighbour: chunks of 300 atoms that hold no bond, between others and at the end
        late = i >= 512
        i, j = i + 700 * late, j + 700 * (j >= 512)
        types = np.concatenate([types[:512], rng.integers(1, 3, 700).astype(np.int32), types[512:], np.ones(700, np.int32)])
    offset = np.concatenate([[0], np.cumsum(np.bincount(i, minlength=len(types)))]).astype(np.int64)
    assert len(j) > 32768
    return types, offset, j.astype(np.int32), rij


_oracle = {}


@pytest.fixture
def shared_from_one_bond(monkeypatch):
    monkeypatch.setenv("GRACE_HIP_PAIR_ROWS", "1")


@pytest.mark.parametrize("model,precision,shared", [("mix2", 64, True), ("mix2", 32, False), ("l2mix", 64, True), ("l2mix", 32, True)])
def test_rows_are_shared_where_the_search_is_worth_it(model_dir, model, precision, shared):
    """85 574 listed bonds on 256 CUs: above the lines of one network in fp64 (49 152) and of two in either precision (24 576,
    49 152), below that of one network in fp32 (98 304)"""
    types, offset, j, rij = _list("long")
    eng = kk.Engine(kk.Model(cases.model_file(model_dir, model)), ["Mo", "W"], precision)
    eng.compute(types, offset, j, rij=rij)
    assert (eng.radial_rows() < eng.edge_count()) == shared


@pytest.mark.parametrize("precision,chunk", [(64, 0), (32, 0), (64, 300)])
@pytest.mark.parametrize("variant", ["plain", "holes", "twice", "rounded", "apart", "long", "gas"])
@pytest.mark.parametrize("model", ["mix2", "l2mix"])
def test_shared_rows_equal_the_oracle(model_dir, shared_from_one_bond, model, variant, precision, chunk):
    _check(model_dir, model, variant, precision, chunk)


@pytest.mark.parametrize("precision,chunk", [(64, 0), (32, 0), (64, 300)])
@pytest.mark.parametrize("variant", ["plain", "long"])
def test_shared_rows_of_wide_models(model_dir, shared_from_one_bond, variant, precision, chunk):
    """64 padded channels: the vector kernel of the A basis, four column blocks in the bond reverse"""
    _check(model_dir, "ch48", variant, precision, chunk)


@pytest.mark.parametrize("precision,chunk", [(64, 0), (32, 0), (64, 300)])
@pytest.mark.parametrize("variant", ["holes", "long"])
def test_shared_rows_of_the_vector_pair_kernels(model_dir, shared_from_one_bond, monkeypatch, variant, precision, chunk):
    """the reverse pair kernel without matrix instructions, which models of more than 128 channels take"""
    monkeypatch.setenv("GRACE_HIP_PAIR_MFMA", "0")
    _check(model_dir, "l2mix", variant, precision, chunk)


@pytest.mark.parametrize("model,species", [("config1", ["W"]), ("config3", ["Al", "Co", "Ni", "Ti"])])
def test_shared_rows_beyond_32_bit_offsets(model_dir, model, species):
    """one pass over 14 M bonds, whose rows of 160 values hold more than 2^31, against the same structure in chunks whose rows hold
    fewer; both at the fp32 gate of the reference (a bond that a chunk cuts has two rows, whose arguments differ in rounding)"""
    pos, cell = synth.bcc_supercell(2.4, 38)
    pos = synth.jitter(pos, 0.05, 6)
    types = np.random.default_rng(6).integers(1, len(species) + 1, len(pos)).astype(np.int32)
    out = {}
    for chunk in (0, 32768):
        s = kk.System(kk.Model(cases.model_file(model_dir, model)), species, skin=0.0, chunksize=chunk, precision=32)
        out[chunk] = s.compute(types, pos, cell, [True] * 3, energies=True)
        bonds, rows = s.engine.edge_count(), s.engine.radial_rows()
        assert bonds * 160 > 2**31 and (rows == bonds / 2 if chunk == 0 else bonds / 2 < rows < bonds)
    cases.check_against(out[0], out[32768], len(pos), 1e-6, 2e-5, 1e-5, 1e-5)


def _check(model_dir, model, variant, precision, chunk):
    path = cases.model_file(model_dir, model)
    types, offset, j, rij = _list(variant)
    eng = kk.Engine(kk.Model(path), ["Mo", "W"], precision)
    eng.set_chunksize(chunk)
    out = eng.compute(types, offset, j, rij=rij, energies=True)
    bonds, rows = eng.edge_count(), eng.radial_rows()
    if variant == "apart":
        assert rows == bonds
    elif chunk or variant == "holes":                 # some bonds have no counterpart in their chunk
        assert bonds / 2 < rows < bonds
    elif variant == "twice":                          # a bond that is listed twice has two rows or, seen from its other end, none
        assert 0.4 * bonds < rows < 0.6 * bonds
    else:
        assert rows == bonds / 2
    if (model, variant) not in _oracle:
        _oracle[(model, variant)] = g1.compute_1l(g1.Model1L(path), types - 1, offset, j, rij) if cases.LAYERS[model] == 1 else \
            g2.compute_2l(g2.Model2L(path), types - 1, offset, j, rij)
    # the bounds of the other parity tests: 1e-10 eV/atom, 1e-9 eV/A in fp64, the fp32 gate of the reference else
    tol = (1e-10, 1e-9, 1e-10, 1e-9) if precision == 64 else (1e-6, 2e-5, 1e-5, 1e-5)
    cases.check_against(out, _oracle[(model, variant)], len(types), *tol)
