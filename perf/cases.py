"""The work whose speed matters to a user of this framework, as cases that can be timed through its public entry points.

Three ways to call the framework are covered, each as its users call it:

* "md"      `System.compute` of a calculator in a molecular dynamics run or a relaxation: host arrays in, energy, forces and
            virial out, the Verlet list kept on the device while the atoms move by less than half the skin;
* "lammps"  `Engine.compute_lammps_device` of a KOKKOS pair style: owned and ghost atoms and the 2-d neighbour view in device
            memory, forces added in place, the list converted anew every LAMMPS_EVERY steps (reneighbouring);
* "batch"   `Batch.compute_device` over many small periodic cells that stay on the device (batched dynamics), work buffers kept;
* "screen"  `Batch.compute` from host arrays, energies only, with the defaults of the class (ranking of candidate cells).

The models are the three benchmark models of this repository (GRACE-1L, 2L and 3L shaped, random weights); sizes run from
one small cell, where launches and the latency of single blocks count, to the largest that three states of fit one GPU.
`precision` is that of the network (geometry, sums and outputs are fp64 always), `tables` the intervals of the radial tables
(0: the radial network itself, the default of the classes; 1024: what the reference's calculator passes on)."""
import functools
import math
import os
import tempfile

import numpy as np
import torch

from grace_runtime_amd import kk, workloads

SKIN = 0.5              # Angstrom, the default of System
LAMMPS_EVERY = 20       # steps between two reneighbourings of a pair style
SPECIES = {"1l": ["W"], "2l": ["Al", "Co", "Ni", "Ti"], "2lb": ["Al", "Ni", "Ti"]}
MODEL_FILE = {"1l": "config1", "2l": "config3", "2lb": "config5", "3l": "config4"}


def _case(name, path, model, size, precision=64, tables=0):
    """size: atoms of a structure, or cells of a batch"""
    return {"name": name, "path": path, "model": model, "size": size, "precision": precision, "tables": tables}


def listed():
    return [
        # GRACE-1L: the smallest supercell one simulates; the benchmark supercell; a large run with the choices of the
        # reference's calculator; a LAMMPS rank of ordinary size whose atom count is no multiple of anything
        _case("1l_md_128", "md", "1l", 128),
        _case("1l_md_8192", "md", "1l", 8192),
        _case("1l_md_65536_f32_tables", "md", "1l", 65536, 32, 1024),
        _case("1l_lammps_4001_tables", "lammps", "1l", 4001, 64, 1024),
        # GRACE-2L: a 3 x 3 x 3 cell with one vacancy; an ordinary run with the calculator's choices; the benchmark alloy
        _case("2l_md_107", "md", "2l", 107),
        _case("2l_md_3999_f32_tables", "md", "2l", 3999, 32, 1024),
        _case("2l_md_32000", "md", "2l", 32000),
        # GRACE-2L over many cells of 32 .. 128 atoms: the benchmark batch on the device; a short list of candidates to rank
        _case("2l_batch_512", "batch", "2lb", 512),
        _case("2l_screen_45_f32", "screen", "2lb", 45, 32),
        # GRACE-3L: a small disordered cell; an ordinary one with the calculator's choices; a large one
        _case("3l_md_96", "md", "3l", 96),
        _case("3l_md_701_f32_tables", "md", "3l", 701, 32, 1024),
        _case("3l_md_3001", "md", "3l", 3001),
    ]


def draw(rng):
    """One more case of the same ranges."""
    path, model, lo, hi = rng.choice([("md", "1l", 128, 65536), ("md", "1l", 128, 65536), ("md", "2l", 100, 32000), ("md", "2l", 100, 32000),
                                      ("md", "3l", 90, 3001), ("md", "3l", 90, 3001), ("lammps", "1l", 1000, 20000), ("batch", "2lb", 8, 512),
                                      ("screen", "2lb", 8, 256)])
    size = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    c = _case("", path, model, size, rng.choice([64, 64, 32]), rng.choice([0, 0, 1024]))
    del c["name"]
    return c


# ---- inputs -------------------------------------------------------------------------------------------------------------

def _lattice(rng, basis, a, atoms):
    """`atoms` sites of the smallest near-cubic supercell that holds them (the rest are vacancies): positions, cell.  `a`: the
    edge, or three edges, of the orthogonal unit cell"""
    a, reps = a * np.ones(3), np.ones(3, dtype=int)
    while reps.prod() * len(basis) < atoms:
        reps[np.argmin(reps * a)] += 1
    grid = np.stack(np.meshgrid(*[np.arange(r) for r in reps], indexing="ij"), -1).reshape(-1, 1, 3)
    sites = (grid + np.asarray(basis)[None]).reshape(-1, 3) * a
    return sites[np.sort(rng.permutation(len(sites))[:atoms])], np.diag(reps * a)


def _structure(model, atoms, rng):
    """positions, cell, 1-based types of one periodic structure"""
    if model == "1l":       # bcc tungsten at a thermal amplitude
        pos, cell = _lattice(rng, [[0, 0, 0], [0.5, 0.5, 0.5]], 3.165, atoms)
        return pos + rng.normal(0.0, 0.05, pos.shape), cell, np.ones(atoms, np.int32)
    if model == "2l":       # fcc alloy of four species
        pos, cell = _lattice(rng, [[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]], 3.6, atoms)
        return pos + rng.normal(0.0, 0.08, pos.shape), cell, rng.integers(1, 5, atoms).astype(np.int32)
    # disordered, eight species, 0.08 atoms / A^3 and no pair closer than 1.8 A: sites of a simple cubic grid (spacing
    # 0.08^(-1/3) = 2.32 A), moved by up to 0.26 A along every axis
    a = 0.08 ** (-1.0 / 3.0)
    pos, cell = _lattice(rng, [[0, 0, 0]], a, atoms)
    return pos + rng.uniform(-0.26, 0.26, pos.shape), cell, rng.integers(1, 9, atoms).astype(np.int32)


HCP = [[0, 0, 0], [0.5, 0.5, 0], [0.5, 5.0 / 6.0, 0.5], [0, 1.0 / 3.0, 0.5]]


def _cells(count, rng):
    """`count` strained and jittered bcc, fcc or hcp cells of 32 .. 128 atoms and three species, as lists (positions, cell,
    types); how many atoms each holds follows from `count` alone"""
    out = []
    for n in np.random.default_rng(count).integers(32, 129, count):
        basis, edge = [([[0, 0, 0], [0.5, 0.5, 0.5]], (1, 1, 1)), ([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]], (1, 1, 1)),
                       (HCP, (1, math.sqrt(3), math.sqrt(8 / 3)))][int(rng.integers(0, 3))]
        pos, cell = _lattice(rng, basis, rng.uniform(2.8, 4.0) * np.array(edge), int(n))
        strain = rng.uniform(-0.03, 0.03, (3, 3))
        deform = np.eye(3) + 0.5 * (strain + strain.T)
        out.append((pos @ deform.T + rng.normal(0.0, 0.1, pos.shape), cell @ deform.T, rng.integers(1, 4, n).astype(np.int32)))
    return out


@functools.lru_cache(maxsize=None)
def _model(key):
    """The loaded model file: what a program keeps for its whole run.  Written once per machine."""
    folder = os.path.join(tempfile.gettempdir(), f"grace_perf_models_{os.getuid()}")
    os.makedirs(folder, exist_ok=True)
    path = os.path.join(folder, MODEL_FILE[key] + ".npz")
    if not os.path.exists(path):
        with tempfile.TemporaryDirectory(dir=folder) as d:
            os.replace(workloads.write_model(MODEL_FILE[key], d), path)
    return kk.Model(path)


def _species(key):
    return SPECIES[key] if key in SPECIES else workloads.config4_species(_model(key).element_names)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    model, species = _model(case["model"]), _species(case["model"])
    opts = {"spline": case["tables"], "precision": case["precision"]}
    if case["path"] in ("batch", "screen"):
        natoms, types, pos, cells, pbc = workloads.batch_arrays(_cells(case["size"], rng))
        s = {"path": case["path"], "batch": kk.Batch(model, species, **opts), "natoms": natoms, "cells": cells, "pbc": pbc}
        if case["path"] == "screen":
            return dict(s, types=types, pos=pos)
        s["batch"].keep_buffers = True
        f64 = {"dtype": torch.float64, "device": "cuda"}
        return dict(s, types=torch.as_tensor(types, device="cuda"), pos=torch.as_tensor(pos, device="cuda"), energy=torch.zeros(len(natoms), **f64),
                    forces=torch.zeros(len(pos), 3, **f64), virial=torch.zeros(len(natoms), 6, **f64))
    pos, cell, types = _structure(case["model"], case["size"], rng)
    pbc = np.array([True, True, True])
    if case["path"] == "md":
        return {"path": "md", "system": kk.System(model, species, SKIN, **opts), "args": (types, pos, cell, pbc)}
    engine = kk.Engine(model, species, case["precision"])
    engine.set_spline(case["tables"])
    return dict(_rank(pos, cell, types, float(engine.cutoff_matrix().max()) + SKIN), path="lammps", engine=engine, step=0)


def _rank(pos, cell, types, reach):
    """One structure as a LAMMPS rank holds it on the device: owned atoms, then their images within `reach`, the full list as
    a 2-d view, the owner of every atom."""
    perm, offset, j, image, shifts = kk.neighbor_search(pos, cell, [True, True, True], reach)
    x, t, n = pos[perm], types[perm], len(pos)
    own = np.flatnonzero(~shifts.any(axis=1))
    key = j.astype(np.int64) * len(shifts) + image
    ghosts = np.unique(key[~np.isin(image, own)])
    gj, gi = ghosts // len(shifts), ghosts % len(shifts)
    index = np.where(np.isin(image, own), j, n + np.searchsorted(ghosts, key)).astype(np.int32)
    count = np.diff(offset)
    nbh = np.zeros((n, int(count.max())), np.int32)
    nbh[np.arange(nbh.shape[1])[None] < count[:, None]] = index
    dev = functools.partial(torch.as_tensor, device="cuda")
    # KOKKOS keeps the view with the atoms running fastest on a GPU
    return {"n": n, "types": dev(np.concatenate([t, t[gj]])), "x": dev(np.concatenate([x, x[gj] + shifts[gi]])), "ilist": dev(np.arange(n, dtype=np.int32)),
            "count": dev(count.astype(np.int32)), "list": dev(nbh).t().contiguous().t(), "owner": dev(np.concatenate([np.arange(n), gj]).astype(np.int32)),
            "forces": torch.zeros(n + len(gj), 3, dtype=torch.float64, device="cuda")}


# ---- one pass -----------------------------------------------------------------------------------------------------------

def run(s):
    if s["path"] == "md":
        return s["system"].compute(*s["args"])
    if s["path"] == "screen":
        return s["batch"].compute(s["natoms"], s["types"], s["pos"], s["cells"], s["pbc"], energy_only=True)
    if s["path"] == "batch":
        s["batch"].compute_device(s["natoms"], s["types"], s["pos"], s["cells"], s["pbc"], s["energy"], s["forces"], s["virial"])
        return s["energy"], s["forces"], s["virial"]
    same, s["step"] = s["step"] % LAMMPS_EVERY != 0, s["step"] + 1
    s["forces"].zero_()
    out = s["engine"].compute_lammps_device(s["n"], s["types"], s["x"], s["ilist"], s["count"], s["list"], owner=s["owner"], forces=s["forces"], same_list=same)
    return out["energy"], s["forces"][:s["n"]], out["virial"]      # with the owner map nothing is added to the ghosts' rows


# ---- what a pass cannot do without --------------------------------------------------------------------------------------

# bonds inside the cutoff per atom; radial networks per pass and their multiply-adds per bond (value and derivative);
# multiply-adds per bond and per atom of the rest, energy and reverse together; bytes of the weights at 64 bits (those
# of the species that are there)
MODEL = {
    "1l": dict(bonds=58, radial=2 * 14848, bond=3 * 25 * 32 * 2, atom=0.9e6, weights=1.5e6),
    "2l": dict(bonds=78, radial=4 * 14848, bond=(3 * 25 * 32 * 2 + 5 * 25 * 32 * 5), atom=1.7e6, weights=3.6e6),
    "2lb": dict(bonds=53.4, radial=4 * 14848, bond=(3 * 25 * 32 * 2 + 5 * 25 * 32 * 5), atom=1.7e6, weights=3.1e6),
    "3l": dict(bonds=71.5, radial=6 * 66560, bond=(3 * 36 * 64 * 2 + 108 * 36 * 64 * 5), atom=70e6, weights=5.5e7),
}


def work(case):
    m = MODEL[case["model"]]
    atoms = case["size"] * (81.4 if case["path"] in ("batch", "screen") else 1)
    # a radial function depends on the distance alone in GRACE-1L and 2L: the two directions of a bond share it; the tables'
    # cubics (value and derivative of 32 or 64 channels per degree) take 6 operations per number
    width = {"1l": 160, "2l": 320, "2lb": 320, "3l": 3 * 384}[case["model"]]
    radial = m["radial"] / (1 if case["model"] == "3l" else 2) if not case["tables"] else 6 * width
    forward = case["path"] == "screen"
    flops = 2.0 * atoms * (m["bonds"] * (radial / (2 if forward else 1) + m["bond"] / (3 if forward else 1)) + m["atom"] / (2 if forward else 1))
    values = 4 + 24 + (0 if forward else 24)        # type and position in, force out
    return {"bytes": atoms * values + m["weights"] * case["precision"] / 64, "flops": flops}


def tolerance(case):
    # largest differences seen over the listed cases, of any output.  64 bits, sums in another order (ordered instead of
    # atomic sums; products, chains and pair reverse by other kernels): 1.9e-14 (the virial of the large GRACE-3L cell, else
    # below 4e-15).  32 bits against 64: 1.8e-6 (forces of GRACE-1L), single values 7.2e-6 of the root mean square.
    return {"rel": 8e-14, "max": 1e-12} if case["precision"] == 64 else {"rel": 8e-6, "max": 3e-5}
