"""The comparison that the tests of the pair kernels rest on (tests/pair_kernels.hip, on the host): a value that is no number, or that
differs where no difference is allowed, is beyond every bound."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("value,wanted,bound,within", [("1", "1", "1e-10", True), ("1.5", "1", "1", True), ("1", "1", "0", True), ("2.5", "1", "1", False),
                                                       ("1", "2", "0", False), ("nan", "1", "1e-10", False), ("nan", "0", "0", False),
                                                       ("1", "nan", "1", False), ("inf", "1", "1e-10", False), ("-inf", "0", "0", False)])
def test_what_is_within_a_bound(value, wanted, bound, within):
    exe, source = os.path.join(ROOT, "tests", "build", "pair_kernels"), os.path.join(ROOT, "tests", "pair_kernels.hip")
    if not os.path.exists(exe) or os.path.getmtime(exe) < os.path.getmtime(source):
        sys.path.insert(0, ROOT)
        import __graft_entry__
        exe = __graft_entry__.build_pair_kernels()
    r = subprocess.run([exe, "compare", value, wanted, bound], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    assert (float(r.stdout) <= 1.0) == within
