"""k_radial_few, which shares a tile of 16 bonds among the waves of a block where there are few tiles, against k_radial: the same
sums in the same order, so every value agrees in every bit whatever number of bonds a call has (radial MLP:
libgrace/include/grace/radial_x.h:11-60)."""
import os
import subprocess
import sys

import numpy as np
import pytest

import cases
from grace_runtime_amd import kk, synth

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def wide(path):
    """hidden width 96: the form of 128, two radial channel blocks"""
    synth.save_model(path, synth.random_model_1l(lmax=2, n_elements=2, element_names=("Mo", "W"), embedding_size=8, nradbase=10, nradmax=20,
                                                 hidden=96, rho_n_out=7, energy_hidden=16, rcut=5.0, inv_avg_n_neigh=1.0 / 26.0, seed=51))
    return path


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("model,species", [("config1", ["W"]), ("mix2", ["Mo", "W"]), ("ch48", ["Mo", "W"]), ("wide", ["Mo", "W"])])
def test_few_and_many_bonds_give_the_same_bits(model_dir, tmp_path, model, species, precision):
    path = wide(str(tmp_path / "wide.npz")) if model == "wide" else cases.model_file(model_dir, model)
    m = kk.Model(path)
    engine = kk.Engine(m, species, precision)
    rng = np.random.default_rng(3)
    line = 16 * (2 if model == "wide" else 3) * 256    # up to here the waves of a block share a tile (256 CUs)
    x = rng.uniform(0.02, 1.0, 2 * line + 5)
    mu = rng.integers(0, len(m.element_names), len(x)).astype(np.int32)
    R, dR = engine.debug_radial(x, mu)
    for n in (1, 15, 16, 17, 255, 16 * 256 + 1, line):
        r, dr = engine.debug_radial(x[:n], mu[:n])
        assert np.array_equal(r, R[:n]) and np.array_equal(dr, dR[:n])


@pytest.mark.parametrize("hidden", [64, 128])
@pytest.mark.parametrize("precision", [64, 32])
def test_species_form_gives_the_same_bits(precision, hidden):
    """the networks of GRACE-3L, launched by themselves (tests/radial_kernels.hip): with ordered sums a chunk of a structure is to give
    the same rows on either side of the line between the two kernels"""
    exe = os.path.join(ROOT, "tests", "build", "radial_kernels")
    if not os.path.exists(exe):
        sys.path.insert(0, ROOT)
        import __graft_entry__
        exe = __graft_entry__.build_kernel_program("radial_kernels")
    r = subprocess.run([exe, str(precision), str(hidden)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert int(r.stdout) == 0
