"""Registers of the built kernels, from the metadata of the code objects in libgrace_hip.so: the job GEMMs keep their operands
and sums in registers (a form of k_gemm_wide that spilled 75 of them was 1.5 times as slow as the one before it), and the
kernels of bonds with a row of their own hold nothing of the paired rows."""
import os
import re
import struct
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "grace_runtime_amd", "libgrace_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """the gfx950 code objects of every offload bundle: 64-bit count, then offset, size and name length of each entry"""
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(n if n < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            pos += 24
            name = data[pos:pos + length]
            pos += length
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{mangled kernel name: (vector registers, of which spilled)}"""
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    out = {}
    with open(LIB, "rb") as f:
        data = f.read()
    for q, obj in enumerate(_code_objects(data)):
        path = tmp_path_factory.mktemp("co") / f"{q}.co"
        path.write_bytes(obj)
        text = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        # one "- .agpr_count: ..." entry per kernel, its keys in alphabetical order
        for entry in re.split(r"\n\s*- \.agpr_count:", text)[1:]:
            name = re.search(r"\.symbol:\s+'?([\w.]+?)\.kd'?\s", entry)
            used, count = re.search(r"\.vgpr_count:\s+(\d+)", entry), re.search(r"\.vgpr_spill_count:\s+(\d+)", entry)
            if name and used and count:
                out[name.group(1)] = max(out.get(name.group(1), (0, 0)), (int(used.group(1)), int(count.group(1))))
    return out


@pytest.mark.parametrize("kernel,forms", [("k_gemm_wide", 2), ("k_gemm_few", 30), ("k_gemm_jobs", 30)])
def test_job_gemms_do_not_spill(kernels, kernel, forms):
    found = {n: spilled for n, (_, spilled) in kernels.items() if re.search(rf"\d{kernel}I[df]", n)}
    assert len(found) >= forms, f"{len(found)} kernels named {kernel} in the library"
    assert not {n: c for n, c in found.items() if c}


# RowsOf::bonds, RowsOf::pairs as template arguments
OWN, PAIRED = "LNS_6RowsOfE0E", "LNS_6RowsOfE2E"


def _three_waves(name):
    """forms of k_bond_bwd that are compiled for three waves per SIMD, 168 registers: fp32, up to 32 channels, up to lmax 4, paired
    rows and tables"""
    m = re.search(r"k_bond_bwdIfLi(\d)ELi(\d)ELNS_6RowsOfE([12])E", name)
    return bool(m) and int(m.group(1)) <= 2 and int(m.group(2)) <= 5


# both forms left to the compiler; those compiled for three waves are held to 168 registers (below)
@pytest.mark.parametrize("kernel,forms", [("k_bond_bwd", 32), ("k_scatter_a_mfma", 28)])
def test_rows_of_their_own_cost_nothing_of_the_paired_rows(kernels, kernel, forms):
    """the paired form keeps the species weights of a lane's bonds beside its operands; the other form must not (GRACE-3L never
    pairs)"""
    own = {n: k for n, k in kernels.items() if re.search(rf"\d{kernel}I[df]", n) and OWN in n and not _three_waves(n.replace(OWN, PAIRED))}
    assert len(own) == forms
    more = [sum(kernels[n.replace(OWN, PAIRED)]) - sum(k) for n, k in own.items()]
    assert min(more) >= 0 and np.median(more) > 0


def test_kernels_of_three_waves_per_simd(kernels):
    """512 registers of a SIMD's lane hold three waves of 168; the forms that spill for it are those whose times are known"""
    bond = {n: k for n, k in kernels.items() if _three_waves(n)}
    tab = {n: k for n, k in kernels.items() if re.search(r"k_scatter_a_tabIf", n)}
    assert len(bond) == 20 and len(tab) == 14
    assert all(used <= 168 for used, _ in [*bond.values(), *tab.values()])
    spilled = {re.search(r"\d(k_[a-z_]+)If((?:Li\dE)+)", n).groups(): s for n, (_, s) in [*bond.items(), *tab.items()] if s}
    assert set(spilled) == {("k_bond_bwd", "Li2ELi5E"), ("k_scatter_a_tab", "Li5ELi2E"), ("k_scatter_a_tab", "Li7ELi1E")}
    assert max(spilled.values()) <= 18


def test_listed_radial_rows_are_a_form_of_their_own(kernels):
    """k_radial without a list holds the species weights, with one it holds neither them nor, without, the list"""
    own = {n: k for n, k in kernels.items() if re.search(r"\d8?k_radialI[df]Li[48]ELi[01]ELi0ELb[01]ELb0EE", n)}
    assert len(own) == 16
    for n, (used, spilled) in own.items():
        assert sum(kernels[n.replace("ELb0EEEv", "ELb1EEEv")]) < used + spilled, n
