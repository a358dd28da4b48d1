"""The groups in which k_groups_fwd and k_groups_bwd walk a sparse matrix, played through on the CPU as the two kernels do:
every output is written once, every row is written before it is added to, and both products are those of the matrix."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("lincomb") / "lincomb_groups")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", os.path.join(HERE, "lincomb_groups.cpp"), "-o", out], check=True)
    return out


def _matrix(kind, rng):
    if kind == "empty":
        return np.zeros((5, 3))
    if kind == "one":
        return np.array([[2.0]])
    if kind == "dense":             # one part of more outputs than a group holds: cut by outputs, rows without terms left over
        W = np.zeros((45, 20))
        W[:40, :17] = rng.integers(1, 9, (40, 17))
        return W
    W = np.zeros((130, 60))         # parts of 1 .. 6 outputs, one of 7 and one of 13 in between, scattered over rows and columns
    r0 = c0 = 0
    for nr, nc in [(1, 1), (9, 6), (33, 3), (2, 7), (5, 2), (20, 13), (3, 1), (4, 4), (12, 5), (1, 6)]:
        W[r0:r0 + nr, c0:c0 + nc] = rng.integers(1, 9, (nr, nc)) * (rng.random((nr, nc)) < 0.7)
        r0, c0 = r0 + nr, c0 + nc
    return W[rng.permutation(130)][:, rng.permutation(60)]


@pytest.mark.parametrize("kind", ["empty", "one", "dense", "parts"])
def test_groups_cover_the_matrix(exe, kind):
    rng = np.random.default_rng(3)
    W = _matrix(kind, rng)
    nrow, nout = W.shape
    r, f = np.nonzero(W)
    text = f"{nrow} {nout} {len(r)}\n" + "".join(f"{a} {b} {W[a, b]}\n" for a, b in zip(r, f))
    lines = [ln.split() for ln in subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.splitlines()]
    groups = [[int(x) for x in ln[1:]] for ln in lines if ln[0] == "group"]
    rows = [(int(ln[1]), int(ln[2]), np.array(ln[3:], float)) for ln in lines if ln[0] == "row"]
    x, g = rng.integers(-9, 9, nrow).astype(float), rng.integers(-9, 9, nout).astype(float)
    fwd, bwd, job_of_row = np.full(nout, np.nan), np.full(nrow, np.nan), np.full(nrow, -1)
    end = 0
    for job, t0, t1, t2, no, *out in groups:
        assert t0 == end and t0 <= t1 <= t2 and no <= 6
        end = t2
        acc = sum((rows[t][2] * x[rows[t][0]] for t in range(t0, t1)), np.zeros(6))
        for o in range(no):
            assert np.isnan(fwd[out[o]])
            fwd[out[o]] = acc[o]
        for t in range(t0, t2):
            a, again, w = rows[t]
            assert np.isnan(bwd[a]) != bool(again)
            assert again == 0 or job_of_row[a] == job       # the wave that wrote it
            job_of_row[a] = job
            bwd[a] = (bwd[a] if again else 0.0) + (w @ g[out] if t < t1 else 0.0)
    assert end == len(rows)
    assert np.array_equal(fwd, W.T @ x) and np.array_equal(bwd, W @ g)
