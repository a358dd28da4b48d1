"""The kernels of the message layers' pair sums by themselves (k_pair_fwd, k_pair_bwd_mfma), every value against the same sums in
fp64 on the host: channel counts that fill a wave or part of one, slots that leave a wave partly empty, atoms with no bond and
with bonds around the chunk sizes, rows per bond and per pair of atoms, every lmax (atom_scatter, bond_scatter_bwd_t,
bond_yi_bwd_g: libgrace/include/grace/fused_cpu.h:836-942,947-1025).  The bound of a value is the length of its longest chain of
additions times the rounding of the type times the sum of the absolute terms (tests/pair_kernels.hip)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def program():
    exe = os.path.join(ROOT, "tests", "build", "pair_kernels")
    if not os.path.exists(exe):
        sys.path.insert(0, ROOT)
        import __graft_entry__
        exe = __graft_entry__.build_pair_kernels()
    return exe


@pytest.mark.parametrize("nl", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("kernel", ["fwd", "bwd"])
def test_pair_kernel_equals_the_sums_of_the_host(program, kernel, precision, nl):
    r = subprocess.run([program, kernel, str(precision), str(nl)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    assert float(r.stdout) <= 1.0
