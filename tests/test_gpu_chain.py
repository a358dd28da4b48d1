"""The fused dense chain of the GRACE-1L / 2L engines (grace_runtime_amd/csrc/jit_chain.hpp: A -> A1 -> AA -> AA1 / AA2 ->
AAA / AAAA as one generated kernel per direction; stage order of the reference, libgrace/src/fused_1l.cpp:260-349)
through the C ABI: against the CPU oracle, and against the same engine with the chain run stage by stage
(GRACE_HIP_CHAIN=0 at engine creation), for the model shapes the generator distinguishes: with and without the AAAA
stage, the legacy product AAA = AA1 x A, channel widths padded to 32, one and two elements, atom counts that do not fill
the last block of atoms, chunked passes, energy-only passes.  Needs an MI355X."""
import os

import numpy as np
import pytest

import cases
from grace_runtime_amd import kk
from oracle import grace_oracle as g1

pytestmark = pytest.mark.gpu

CASES = [("config1", "config1"), ("ch20", "alloy54"), ("ch3", "triclinic"), ("chleg", "alloy54"), ("ch20", "molecule")]


def _engine(path, species, precision, fused):
    old = os.environ.get("GRACE_HIP_CHAIN")
    os.environ["GRACE_HIP_CHAIN"] = "1" if fused else "0"
    try:
        return kk.Engine(kk.Model(path), species, precision)
    finally:
        if old is None:
            del os.environ["GRACE_HIP_CHAIN"]
        else:
            os.environ["GRACE_HIP_CHAIN"] = old


def _stages(eng):
    eng.set_profile(True)
    eng.run()
    names = set(eng.stage_times())
    eng.set_profile(False)
    return names


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model,struct", CASES)
def test_fused_chain_equals_the_oracle_and_the_staged_chain(model_dir, model, struct, precision):
    path = cases.model_file(model_dir, model)
    om = g1.Model1L(path)
    species = [s.decode() for s in om.d["element_names"]]
    pos, cell, pbc, types = cases.STRUCTURES[struct]()
    types = np.minimum(types, om.n_elements).astype(np.int32)
    rc = float(np.max(om.cut))
    pcell, shift = kk._padded_cell_arrays(cell, pos, rc, pbc)
    perm, offset, j, image, shifts = kk.neighbor_search(pos + shift, pcell, pbc, rc)
    rij = cases.bond_vectors(pos, perm, offset, j, image, shifts)
    n = len(pos)
    ref = g1.compute_1l(om, types[perm] - 1, offset, j, rij)
    fused, staged = _engine(path, species, precision, True), _engine(path, species, precision, False)
    out = {}
    for tag, eng in (("fused", fused), ("staged", staged)):
        eng.upload(types[perm], offset, j, rij=rij)
        names = _stages(eng)
        assert ("chain_fwd" in names and "chain_bwd" in names and "fc_AA1" not in names) == (tag == "fused"), (tag, sorted(names))
        eng.run(energies=True)
        out[tag] = eng.fetch(energies=True)
    fs = max(1.0, np.abs(ref["forces"]).max())
    tol = (1e-10, 1e-9, 1e-9) if precision == 64 else (1e-6, 2e-5, 1e-5)
    for tag in ("fused", "staged"):
        o = out[tag]
        assert abs(o["energy"] - ref["energy"]) / n < tol[0] * fs, tag
        assert np.abs(o["forces"] - ref["forces"]).max() < tol[1] * fs, tag
        assert np.abs(o["energies"] - ref["energies"]).max() < tol[0] * fs, tag
        assert np.abs(o["virial"] - ref["virial"]).max() < tol[2] * max(1.0, np.abs(ref["virial"]).max()), tag
    # the two ways through the chain differ in summation order only
    same = 1e-11 if precision == 64 else 2e-5
    assert abs(out["fused"]["energy"] - out["staged"]["energy"]) / n < same * fs
    assert np.abs(out["fused"]["forces"] - out["staged"]["forces"]).max() < 10 * same * fs
    # energy-only pass and a pass in chunks that cut the blocks of atoms
    fused.run(energy_only=True)
    assert abs(fused.fetch()["energy"] - ref["energy"]) / n < tol[0] * fs
    fused.set_chunksize(13)
    fused.run(energies=True)
    o = fused.fetch(energies=True)
    assert fused.chunksize == 13
    assert abs(o["energy"] - ref["energy"]) / n < tol[0] * fs and np.abs(o["forces"] - ref["forces"]).max() < tol[1] * fs
    fused.close()
    staged.close()


def test_models_outside_the_generator_keep_the_staged_chain(model_dir):
    """channel widths other than 32 (the fixture models of the reference: 16; mix2: 32 and 64) run stage by stage"""
    for name, fixture, species in (("grace_1l_order3", True, ["Mo", "W"]), ("mix2", False, ["Mo", "W"])):
        path = os.path.join(cases.REF_FIXTURES, name + ".npz") if fixture else cases.model_file(model_dir, name)
        eng = kk.Engine(kk.Model(path), species, 64)
        pos, cell, pbc, types = cases.structure_alloy54()
        perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, pbc, 5.0)
        eng.upload(types[perm], offset, j, positions=pos[perm], image=image, shifts=shifts)
        names = _stages(eng)
        assert "chain_fwd" not in names and "fc_A1" in names
        eng.close()


def test_compiled_kernels_are_kept_on_disk_for_the_next_process(model_dir, tmp_path):
    """GRACE_HIP_CACHE: the first process compiles the generated kernels and leaves their code objects in the directory, the
    second one loads them (no compiler run: engine creation in a fraction of the time) and computes the same numbers"""
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    path = cases.model_file(model_dir, "ch20")
    code = (
        "import sys, time, numpy as np\n"
        f"sys.path.insert(0, {root!r}); sys.path.insert(0, {os.path.join(root, 'tests')!r})\n"
        "import cases\n"
        "from grace_runtime_amd import kk\n"
        "t = time.perf_counter()\n"
        f"eng = kk.Engine(kk.Model({path!r}), ['Mo', 'W'], 64)\n"
        "dt = time.perf_counter() - t\n"
        "pos, cell, pbc, types = cases.structure_alloy54()\n"
        "perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, pbc, 5.0)\n"
        "out = eng.compute(types[perm], offset, j, positions=pos[perm], image=image, shifts=shifts)\n"
        "print(dt, repr(out['energy']), repr(float(np.abs(out['forces']).sum())))\n")
    env = dict(os.environ, GRACE_HIP_CACHE=str(tmp_path / "cache"))
    runs = []
    for _ in range(2):
        res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env, timeout=300)
        assert res.returncode == 0, res.stderr
        runs.append(res.stdout.strip().split("\n")[-1].split())
    files = os.listdir(tmp_path / "cache")
    assert len(files) >= 3 and all(f.endswith(".co") for f in files)          # three products and the chain
    assert float(runs[1][0]) < 0.5 * float(runs[0][0])
    assert abs(float(runs[0][1]) - float(runs[1][1])) < 1e-9 * abs(float(runs[0][1]))
    assert abs(float(runs[0][2]) - float(runs[1][2])) < 1e-9 * abs(float(runs[0][2]))
    # a file that the driver does not load (cut short here) is dropped, its source compiled again and the file replaced
    sizes = {f: os.path.getsize(tmp_path / "cache" / f) for f in files}
    for f in files:
        with open(tmp_path / "cache" / f, "r+b") as fh:
            fh.truncate(200)
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env, timeout=300)
    assert res.returncode == 0, res.stderr
    third = res.stdout.strip().split("\n")[-1].split()
    assert abs(float(third[1]) - float(runs[0][1])) < 1e-9 * abs(float(runs[0][1]))
    assert {f: os.path.getsize(tmp_path / "cache" / f) for f in os.listdir(tmp_path / "cache")} == sizes
    # switched off: nothing is written
    env0 = dict(os.environ, GRACE_HIP_CACHE="0", HOME=str(tmp_path / "home"))
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env0, timeout=300)
    assert res.returncode == 0, res.stderr
    assert not os.path.exists(tmp_path / "home" / ".cache" / "grace_hip")


@pytest.mark.parametrize("model,species,precision,fused,files", [("config3", ["Al", "Co", "Ni", "Ti"], 64, "1", 2), ("l2ord4", ["Mo", "W"], 64, "1", 2),
                                                                 ("l2deep", ["Mo", "W"], 32, "1", 4), ("config3", ["Al", "Co", "Ni", "Ti"], 64, "0", 4),
                                                                 ("l2ord4", ["Mo", "W"], 64, "0", 6)])
def test_a_two_layer_engine_compiles_what_a_pass_launches(model_dir, tmp_path, model, species, precision, fused, files):
    """the code objects that creating an engine leaves on disk: the chain of each layer, with the third product of a chain that leaves
    it outside, or without chains all products of both layers"""
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = (f"import sys; sys.path.insert(0, {root!r})\n"
            "from grace_runtime_amd import kk\n"
            f"kk.Engine(kk.Model({cases.model_file(model_dir, model)!r}), {species!r}, {precision})\n")
    env = dict(os.environ, GRACE_HIP_CACHE=str(tmp_path), GRACE_HIP_CHAIN=fused)
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env=env, timeout=110)
    assert res.returncode == 0, res.stderr
    assert len(os.listdir(tmp_path)) == files


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("natoms", [9, 350, 1020, 1030])
@pytest.mark.parametrize("model", ["ch20", "config3"])
def test_chain_in_parts(model_dir, model, natoms, precision):
    """few atoms: the groups of the chain dealt to 2 .. 8 blocks (jit_chain.hpp: chain_fwd_part, chain_bwd_part, k_chain_sum);
    256 CUs hold 8 parts up to 256 atoms, 2 parts up to 1024, one block per 8 atoms above"""
    from grace_runtime_amd import synth
    from oracle import grace_oracle_2l as g2
    path = cases.model_file(model_dir, model)
    om = g1.Model1L(path) if model == "ch20" else g2.Model2L(path)
    pos, cell = synth.bcc_supercell(3.165, 9)
    rng = np.random.default_rng(natoms)
    pos = synth.jitter(pos, 0.05, 3)[np.sort(rng.permutation(len(pos))[:natoms])]      # dilute: the atoms stay in the full box
    types = rng.integers(1, om.n_elements + 1, natoms).astype(np.int32)
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True] * 3, float(np.max(om.cut)))
    rij = cases.bond_vectors(pos, perm, offset, j, image, shifts)
    species = [s.decode() for s in om.d["element_names"]]
    eng = _engine(path, species, precision, True)
    eng.set_profile(True)
    out = eng.compute(types[perm], offset, j, rij=rij, energies=True)
    sums = {s for s in eng.stage_times() if s.startswith("chain_sum")}
    assert sums == (set() if natoms > 1024 else {"chain_sum"} if model == "ch20" else {"chain_sum_L1", "chain_sum_L2"})
    ref = (g1.compute_1l if model == "ch20" else g2.compute_2l)(om, types[perm] - 1, offset, j, rij)
    cases.check_against(out, ref, natoms, *((1e-10, 1e-9, 1e-10, 1e-9) if precision == 64 else (1e-6, 2e-5, 1e-5, 1e-5)))


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("natoms", [1025, 2041, 4105])
def test_blocks_that_share_a_cu(model_dir, natoms, precision):
    """the whole form of both chains of GRACE-2L, whose paths are handed over in pieces of four to six functions and whose rows of
    X0 take turns in layer 2, against the stages: one block per CU, the last one of a single atom; one CU without a block; twice
    as many blocks as CUs and one.  The two differ in the order in which 64 terms are added, which moves a sum by at most 64 eps
    of its terms (1.4e-14, 7.6e-6); forces come through both layers, both ways, and get ten times the bound of the energies."""
    from grace_runtime_amd import synth
    from oracle import grace_oracle_2l as g2
    path = cases.model_file(model_dir, "config3")
    pos, cell = synth.bcc_supercell(3.165, 13)
    rng = np.random.default_rng(natoms)
    pos = synth.jitter(pos, 0.05, 3)[np.sort(rng.permutation(len(pos))[:natoms])]
    om = g2.Model2L(path)
    types = rng.integers(1, om.n_elements + 1, natoms).astype(np.int32)
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True] * 3, float(np.max(om.cut)))
    rij = cases.bond_vectors(pos, perm, offset, j, image, shifts)
    species = [s.decode() for s in om.d["element_names"]]
    out = []
    for fused in (True, False):
        eng = _engine(path, species, precision, fused)
        eng.set_profile(True)
        out.append(eng.compute(types[perm], offset, j, rij=rij, energies=True))
        assert ("chain_bwd_L2" in eng.stage_times()) == fused
    same = 1e-11 if precision == 64 else 2e-5
    cases.check_against(out[0], out[1], natoms, same, 10 * same, same, 10 * same)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model", ["l2ord4", "l2deep"])
def test_third_product_of_many_outputs(model_dir, model, precision):
    """l2ord4: P3 path by path together with the fourth-order stage, whose values stay in registers (layer 1); l2deep: the paths of
    l = 5 are cut at nine functions and an output is fed by both parts, so P3 stays outside of the chain kernels (both layers in
    fp32; in fp64 the rows of layer 2 do not fit the LDS and it runs stage by stage).  In parts (9 and 250 atoms) and whole (1030),
    against the oracle and against the stages, bounds as above."""
    from grace_runtime_amd import synth
    from oracle import grace_oracle_2l as g2
    path = cases.model_file(model_dir, model)
    om = g2.Model2L(path)
    engines = [_engine(path, ["Mo", "W"], precision, fused) for fused in (True, False)]
    same = 1e-11 if precision == 64 else 2e-5
    for natoms in (9, 250, 1030):
        pos, cell = synth.bcc_supercell(3.165, 9)
        rng = np.random.default_rng(natoms)
        pos = synth.jitter(pos, 0.05, 3)[np.sort(rng.permutation(len(pos))[:natoms])]
        types = rng.integers(1, 3, natoms).astype(np.int32)
        perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True] * 3, float(np.max(om.cut)))
        rij = cases.bond_vectors(pos, perm, offset, j, image, shifts)
        out = []
        for eng in engines:
            eng.set_profile(True)
            out.append(eng.compute(types[perm], offset, j, rij=rij, energies=True))
        names = set(engines[0].stage_times())
        chains = {"_L1"} if model == "l2deep" and precision == 64 else {"_L1", "_L2"}
        assert {s[9:] for s in names if s.startswith("chain_bwd")} == chains
        # the 71 functions of layer 2 of l2deep are more than a chain in parts keeps track of
        assert {s[9:] for s in names if s.startswith("chain_sum")} == (set() if natoms > 1024 else chains if model == "l2ord4" else {"_L1"})
        assert all((f"prod_3{t}" in names and f"prod_3_bwd{t}" in names) == (model == "l2deep") for t in chains)
        cases.check_against(out[0], out[1], natoms, same, 10 * same, same, 10 * same)
        if natoms <= 250:
            ref = g2.compute_2l(om, types[perm] - 1, offset, j, rij)
            cases.check_against(out[0], ref, natoms, *((1e-10, 1e-9, 1e-10, 1e-9) if precision == 64 else (1e-6, 2e-5, 1e-5, 1e-5)))
