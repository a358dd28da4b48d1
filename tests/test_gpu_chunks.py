"""Atom chunking of an engine pass (System(chunksize=...), python/kk/kk_api.h:72-75,86): a structure evaluated in chunks of
atoms equals the one-pass result for GRACE-1L, 2L and 3L; the automatic choice follows the memory the library may use; an
allocation failure halves the chunk."""
import contextlib
import os
import re

import numpy as np
import pytest

import cases
from grace_runtime_amd import _lib, kk, workloads
from test_gpu_paired_rows import _list as bond_list

pytestmark = pytest.mark.gpu


def _same(a, b, n, tol=1e-10):
    fs = max(1.0, np.abs(b["forces"]).max())
    assert abs(a["energy"] - b["energy"]) / n < tol * fs
    assert np.abs(a["forces"] - b["forces"]).max() < 10 * tol * fs
    assert np.abs(a["virial"] - b["virial"]).max() < 100 * tol * fs
    if "energies" in b:
        assert np.abs(a["energies"] - b["energies"]).max() < tol * fs


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model,struct,species", [("mix2", "alloy54", ["Mo", "W"]), ("cut2", "slab", ["Al", "Ni"]), ("config1", "config1", ["W"]),
                                                  ("l2mix", "alloy54", ["Mo", "W"]), ("l2mix", "slab", ["Mo", "W"]), ("config3", "fcc108", ["Al", "Co", "Ni", "Ti"]),
                                                  ("l3mix", "alloy54", ["Mo", "W"]), ("l3wide", "fcc108", ["Al", "Ni"]), ("l3el", "alloy54", ["Mo", "W"])])
def test_chunked_pass_equals_one_pass(model_dir, model, struct, species, precision):
    """chunk sizes that split the tiles of 16 atoms of one element, a chunk of one atom, a chunk larger than the structure"""
    pos, cell, pbc, types = cases.STRUCTURES[struct]()
    types = np.minimum(types, len(species)).astype(np.int32)
    n = len(pos)
    m = kk.Model(cases.model_file(model_dir, model))
    one = kk.System(m, species, skin=0.0, chunksize=0, precision=precision)
    ref = one.compute(types, pos, cell, pbc, energies=True)
    assert one.chunksize == 0
    tol = 1e-10 if precision == 64 else 2e-6
    for cs in (7, 16, 21, 1, n - 1, n, 5 * n):
        s = kk.System(m, species, skin=0.0, chunksize=cs, precision=precision)
        out = s.compute(types, pos, cell, pbc, energies=True)
        assert s.chunksize == (cs if cs < n else 0)
        _same(out, ref, n, tol)
        again = s.compute(types, pos + 1e-3, cell, pbc, energies=True)          # a second call reuses the chunk layout
        _same(again, one.compute(types, pos + 1e-3, cell, pbc, energies=True), n, tol)
        del s


@pytest.mark.parametrize("model", ["uq2", "uq2l", "uq3l"])
def test_chunked_uq_and_energy_only(model_dir, model):
    pos, cell, pbc, types = cases.structure_alloy54()
    m = kk.Model(cases.model_file(model_dir, model))
    ref = kk.System(m, ["Mo", "W"], skin=0.0, chunksize=0).compute(types, pos, cell, pbc, uq=True, energies=True)
    s = kk.System(m, ["Mo", "W"], skin=0.0, chunksize=13)
    out = s.compute(types, pos, cell, pbc, uq=True, energies=True)
    _same(out, ref, len(pos))
    for k in ("gamma", "atomic_sigma"):
        assert np.abs(out[k] / ref[k] - 1).max() < 1e-9
    assert np.array_equal(out["gmm_cluster"], ref["gmm_cluster"])
    eo = s.compute(types, pos, cell, pbc, energy_only=True)
    assert abs(eo["energy"] - ref["energy"]) < 1e-9


@pytest.mark.parametrize("model", ["mix2", "l2mix", "l3mix"])
def test_chunked_batch_equals_one_pass(model_dir, model):
    """several structures in one list, chunks that cut through structures"""
    structs = workloads.structures_config5(6)
    natoms, types, pos, cells, pbc = workloads.batch_arrays(structs)
    types = np.minimum(types, 2).astype(np.int32)
    m = kk.Model(cases.model_file(model_dir, model))
    ref = kk.Batch(m, ["Mo", "W"], chunksize=0).compute(natoms, types, pos, cells, pbc, energies=True)
    b = kk.Batch(m, ["Mo", "W"], chunksize=50)
    out = b.compute(natoms, types, pos, cells, pbc, energies=True)
    fs = max(1.0, np.abs(ref["forces"]).max())
    assert np.abs(out["energy"] - ref["energy"]).max() < 1e-9 * fs
    assert np.abs(out["forces"] - ref["forces"]).max() < 1e-9 * fs
    assert np.abs(out["virial"] - ref["virial"]).max() < 1e-8 * fs
    assert np.abs(out["energies"] - ref["energies"]).max() < 1e-9 * fs


def test_automatic_chunk_follows_the_memory_the_library_may_use(tmp_path):
    """configuration 2 (8192 atoms) under a cap on the library's device memory: the automatic choice splits the structure,
    the result is the one-pass result; a cap that even 512 atoms per pass do not fit is reported, and the engine recovers"""
    pos, cell, pbc, types = workloads.structure_config2()
    m = kk.Model(workloads.write_model("config1", str(tmp_path)))
    L = _lib.lib()
    ref = kk.System(m, ["W"], skin=0.0, chunksize=0).compute(types, pos, cell, pbc)
    s = kk.System(m, ["W"], skin=0.0)                    # chunksize -1: automatic
    out = s.compute(types, pos, cell, pbc)
    assert s.chunksize == 0                              # fits: one pass
    _same(out, ref, len(pos))
    s.release_buffers()
    said = []
    kk.set_logger(lambda level, msg: said.append((level, msg)))
    try:
        s2 = kk.System(m, ["W"], skin=0.0)
        L.gr_set_memory_limit(L.gr_memory_in_use() + 900 * 1024 * 1024)
        out = s2.compute(types, pos, cell, pbc)
        assert s2.chunksize == 1024                      # the largest power of two whose work buffers fit 70 % of 900 MB
        assert any(level == 0 and "chunksize auto: 1024 atoms per pass" in msg for level, msg in said)
        _same(out, ref, len(pos))
        # a fixed chunk that does not fit: reported, not retried
        s2.release_buffers()
        L.gr_set_memory_limit(0)
        s3 = kk.System(m, ["W"], skin=0.0, chunksize=8000)
        L.gr_set_memory_limit(L.gr_memory_in_use() + 900 * 1024 * 1024)
        with pytest.raises(RuntimeError, match="does not fit"):
            s3.compute(types, pos, cell, pbc)
        L.gr_set_memory_limit(L.gr_memory_in_use() + 60 * 1024 * 1024)
        with pytest.raises(RuntimeError, match="does not fit"):
            s2.compute(types, pos, cell, pbc)
        assert any(level == 0 and "chunksize auto: 512 atoms per pass" in msg for level, msg in said)
    finally:
        L.gr_set_memory_limit(0)
        kk.set_logger(None)
    out = s2.compute(types, pos, cell, pbc)              # the engine is usable again
    _same(out, ref, len(pos))


@pytest.mark.parametrize("model", ["mix2", "l2mix"])
def test_automatic_chunk_counts_what_the_paired_rows_keep(model_dir, model):
    """a list whose bonds share radial rows keeps 16 bytes more per bond, and every buffer is allocated an eighth larger: what
    the engine says it keeps, with the radial network and with tables (where no rows are shared)"""
    types, offset, j, rij = bond_list("long")
    L, kept, n = _lib.lib(), {}, len(types)
    said = []
    kk.set_logger(lambda level, msg: said.append(msg))
    try:
        for intervals in (0, 256):
            eng = kk.Engine(kk.Model(cases.model_file(model_dir, model)), ["Mo", "W"], 64)
            eng.set_spline(intervals)
            eng.set_chunksize(-1)
            base = L.gr_memory_in_use()
            eng.compute(types, offset, j, rij=rij)
            work = L.gr_memory_in_use() - base
            eng.release_buffers()
            L.gr_set_memory_limit(L.gr_memory_in_use() + work // 2)
            said.clear()
            with contextlib.suppress(MemoryError, RuntimeError):    # whether 512 atoms per pass fit that is not the matter here
                eng.compute(types, offset, j, rij=rij)
            L.gr_set_memory_limit(0)
            found = [re.search(r"(\d+) MB of work buffers and (\d+) MB kept per 1000 atoms", msg) for msg in said]
            kept[intervals] = [int(m.group(2)) for m in found if m][0]
    finally:
        L.gr_set_memory_limit(0)
        kk.set_logger(None)
    # the message counts whole MB
    assert kept[0] - kept[256] >= 16 * len(j) / n * 1000 / 1048576 - 1 > 0


def test_few_atoms_take_no_more_memory_per_atom(model_dir):
    """GRACE-3L deals the couples of few atoms (below 1408 with 64 channels and 256 CUs) to blocks that leave an adjoint each: in memory
    that the pass holds anyway, which the automatic chunk counts"""
    m, L, held, energy = kk.Model(cases.model_file(model_dir, "config4")), _lib.lib(), {}, {}
    for n in (96, 2880):                                  # dimers: the same bonds per atom
        eng = kk.Engine(m, ["Mo", "W"], 64)
        eng.set_chunksize(0)
        base = L.gr_memory_in_use()
        i = np.arange(n)
        out = eng.compute(1 + i % 2, np.arange(n + 1), i ^ 1, rij=np.where(i % 2, -1.0, 1.0)[:, None] * np.array([1.5, 1.2, 1.0]))
        held[n], energy[n] = L.gr_memory_in_use() - base, out["energy"] / n
        del eng
    assert abs(energy[96] - energy[2880]) < 1e-10
    assert held[96] / 96 < held[2880] / 2880 + 4 * 2 ** 20 / 96        # the parts of the reduces: up to 2 MB; those of the couples took 30


def test_outputs_accumulate_on_request(model_dir):
    """GR_FLAG_ACCUMULATE: the outputs of a call are added to the caller's values (libgrace/include/grace/system.h:66-75)"""
    pos, cell, pbc, types = cases.structure_alloy54()
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, pbc, 5.0)
    eng = kk.Engine(kk.Model(cases.model_file(model_dir, "mix2")), ["Mo", "W"], 64)
    args = dict(positions=pos[perm], image=image, shifts=shifts, energies=True)
    one = eng.compute(types[perm], offset, j, **args)
    two = eng.compute(types[perm], offset, j, add_to=one, **args)
    for k in ("energy", "forces", "virial", "energies"):
        assert np.allclose(two[k], 2.0 * np.asarray(one[k]), rtol=0, atol=1e-11 * max(1.0, np.abs(one[k]).max()))
