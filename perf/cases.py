"""The workloads this engine's speed is measured on.

Each case is a molecular-dynamics job a user runs through the public Python
interface (``HipEngine``, ``HipBatch``, ``NativeWarmStart``): one step at a
time under a host loop, strides of steps at 2 fs, constant pressure, NVE,
force evaluations and minimisations driven from outside, and batches of
replicas.  Sizes follow the benchmark configurations (2.4k, 27k, 100k and 250k
atoms, ensembles of 2k-30k atoms with 32^3-64^3 meshes).

The systems are solvated chains at liquid density: rigid three-site water,
extended hydrocarbon-like strands with constrained C-H bonds, harmonic bonds
and angles, torsions, scaled 1-4 pairs, and a few ions, in rectangular boxes,
truncated octahedra or rhombic dodecahedra.  Waters start hydrogen-bonded (a
diamond-lattice network with random proton order, displaced and turned by
thermal amounts), so 2 fs steps at 300 K are stable from the first one and
nothing has to be equilibrated.

Frames come back as single-precision positions and velocities: what a DCD
frame holds, and the type the engine keeps velocities in.
"""
import math
import os
import sys
from functools import lru_cache

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "making-it-rain-webgpu_amd"))

from mdcore import native  # noqa: E402
from mdcore.engine import HipBatch, HipEngine, RunOptions  # noqa: E402
from mdcore.state import OpenMMState  # noqa: E402
from mdcore.system import (CMMotionRemover, HarmonicAngleForce, HarmonicBondForce, MonteCarloBarostat,  # noqa: E402
                           NonbondedForce, OpenMMSystem, PeriodicTorsionForce, PositionRestraintForce, reduceBox)

KB = 0.008314462618153242      # kJ/mol/K
COULOMB = 138.93545764498457   # kJ nm / mol / e^2
CUTOFF = 1.0
TOLERANCE = 5e-4
DT = 0.002
TEMPERATURE = 300.0
MOLECULES_PER_NM3 = 33.43      # water at 1.0 g/cm^3
LATTICE = (8 / MOLECULES_PER_NM3) ** (1 / 3)  # nm; 8 waters per cubic lattice cell

# the lattice vectors of each cell shape, in lattice cells, per unit of "cells"
SHAPES = {"octahedron": ((1, 1, -1), (-1, 1, -1), (-1, 1, 1)), "dodecahedron": ((1, 1, 0), (1, -1, 0), (1, 0, 1))}


# ---- the cases ------------------------------------------------------------------

def listed():
    return [
        # a host loop that acts between steps (interactive viewers, steered and
        # metadynamics drivers): one 2 fs step, then the frame; the 2.4k-atom
        # system.  Launches and the host path are all there is.
        {"name": "step-2k", "job": "run", "shape": "box", "cells": "5 5 4", "mesh": 32, "steps": 1},
        # production NVT of the same system, a frame every 50 steps
        {"name": "nvt-2k", "job": "run", "shape": "box", "cells": "5 5 4", "mesh": 32, "steps": 50},
        # an NVE stability check (Verlet) of a mid-sized system in an oblong
        # box with the mesh the Ewald tolerance asks for, not a power of two
        {"name": "nve-9k", "job": "run", "shape": "box", "cells": "8 7 7", "mesh": 0, "steps": 50, "verlet": True},
        # production NVT in a truncated octahedron, the protein-ligand size
        {"name": "nvt-31k-octahedron", "job": "run", "shape": "octahedron", "cells": "7", "mesh": 64, "steps": 50},
        # restrained NPT equilibration in a rhombic dodecahedron, a barostat
        # attempt every 25 steps
        {"name": "npt-99k-dodecahedron", "job": "run", "shape": "dodecahedron", "cells": "13", "mesh": 96, "steps": 50,
         "restraint": 1000.0, "barostat": 25},
        # the largest single system: 250k atoms, 128^3 mesh
        {"name": "nvt-243k", "job": "run", "shape": "box", "cells": "22 22 22", "mesh": 128, "steps": 25},
        # forces and energy at positions the caller brings (an external
        # integrator, a rescoring pass)
        {"name": "forces-31k-octahedron", "job": "forces", "shape": "octahedron", "cells": "7", "mesh": 64},
        # the minimiser ahead of a production run
        {"name": "minimise-9k", "job": "minimise", "shape": "box", "cells": "8 7 7", "mesh": 48, "iterations": 10},
        # a small ensemble: eight replicas of the 2.4k-atom system
        {"name": "batch-8x2k", "job": "batch", "shape": "box", "cells": "5 5 4", "mesh": 32, "steps": 50,
         "replicas": 8},
        # the ensemble of the benchmark: 2k-30k atoms, boxes and truncated
        # octahedra alternating, meshes by size
        {"name": "batch-64-mixed", "job": "batch", "shape": "mixed", "cells": "", "mesh": -1, "steps": 20,
         "replicas": 64},
        # the same kind of ensemble with SHAKE started from a network
        {"name": "batch-12-learned", "job": "batch", "shape": "mixed", "cells": "", "mesh": -1, "steps": 20,
         "replicas": 12, "learned": True},
    ]


def draw(rng):
    kind = rng.choice(["step", "nvt", "nvt", "nve", "npt", "forces", "minimise", "batch", "batch"])
    if kind == "batch":
        n = int(round(math.exp(rng.uniform(math.log(2), math.log(48)))))
        same = rng.random() < 0.3
        case = {"job": "batch", "shape": "box" if same else "mixed", "cells": "", "mesh": 0 if same else -1,
                "steps": rng.randint(5, 25), "replicas": n}
        if same:
            a = rng.randint(4, 6)
            case["cells"] = "%d %d %d" % (a + rng.randint(0, 1), a + rng.randint(0, 1), a)
        if rng.random() < 0.3:
            case["learned"] = True
        return case
    shape = rng.choice(["box", "octahedron", "dodecahedron"])
    # 1.5k to 250k atoms, uniform in the logarithm
    largest = {"step": 60e3, "minimise": 60e3, "forces": 120e3}.get(kind, 250e3)
    atoms = math.exp(rng.uniform(math.log(2e3), math.log(largest)))
    if shape == "box":
        a = max(4, int(round((atoms / 24) ** (1 / 3))))
        cells = "%d %d %d" % (a + rng.randint(0, 1 + a // 6), a + rng.randint(0, 1), a)
    elif shape == "octahedron":
        cells = str(max(3, int(round((atoms / 96) ** (1 / 3)))))
    else:
        cells = str(max(4, int(round((atoms / 48) ** (1 / 3)))))
    case = {"job": {"step": "run", "nvt": "run", "nve": "run", "npt": "run"}.get(kind, kind), "shape": shape,
            "cells": cells, "mesh": rng.choice([0, 0, -1])}
    if case["job"] == "run":
        case["steps"] = 1 if kind == "step" else rng.randint(5, 25 if atoms > 60e3 else 60)
    if kind == "nve":
        case["verlet"] = True
    if kind == "npt":
        case["barostat"] = rng.choice([10, 25])
        if rng.random() < 0.5:
            case["restraint"] = 1000.0
    if kind == "minimise":
        case["iterations"] = rng.randint(3, 12)
    return case


def _replicas(case):
    """(shape, cells) of each replica of a batch."""
    if case["shape"] != "mixed":
        return [(case["shape"], case["cells"])] * case["replicas"]
    # 2k-30k atoms, spread evenly over the logarithm, boxes and octahedra in turn
    r = np.random.default_rng(20261202)
    out = []
    for k in range(case["replicas"]):
        atoms = math.exp(math.log(2000) + (k + 0.5) / case["replicas"] * math.log(15))
        if k % 2 == 0:
            a = max(4, int((atoms / 24) ** (1 / 3)))
            c = max(4, int(round(atoms / (24 * a * a))))
            out.append(("box", "%d %d %d" % (a, a, c)))
        else:
            out.append(("octahedron", str(max(3, int(round((atoms / 96) ** (1 / 3)))))))
    order = r.permutation(len(out))
    return [out[k] for k in order]


def _systems(case):
    which = _replicas(case) if case["job"] == "batch" else [(case["shape"], case["cells"])]
    return [_topology(shape, cells, case["mesh"], case.get("restraint", 0.0), case.get("barostat", 0))
            for shape, cells in which]


# ---- the systems -----------------------------------------------------------------

def _cell(shape, cells):
    """The cell's lattice vectors in lattice cells (integers)."""
    n = [int(c) for c in cells.split()]
    return np.diag(n) if shape == "box" else np.array(SHAPES[shape]) * n[0]


def _lattice(M):
    """Oxygen sites (fractional) and the two hydrogen directions of each, for
    the cell with integer lattice vectors M: a diamond lattice where every
    molecule gives two hydrogens and takes two.  Molecules form straight
    zigzag chains in two families; a chain's protons all point one way or
    the other, which any choice per chain keeps consistent."""
    rng = np.random.default_rng(int(abs(np.linalg.det(M))) + 7)
    Q = 4 * M  # quarter cells
    det = int(round(np.linalg.det(Q)))
    adj = np.rint(np.linalg.inv(Q) * det).astype(np.int64) * (1 if det > 0 else -1)
    det = abs(det)

    def scaled(x):  # fractional coordinates times det
        return x @ adj

    corners = np.array([[i, j, k] for i in (0, 1) for j in (0, 1) for k in (0, 1)]) @ M
    lo, hi = corners.min(0) - 1, corners.max(0) + 1
    g = np.stack(np.meshgrid(*[np.arange(a, b) for a, b in zip(lo, hi)], indexing="ij"), -1).reshape(-1, 3)
    fcc = np.array([[0, 0, 0], [0, 2, 2], [2, 0, 2], [2, 2, 0]])
    A = (4 * g[:, None, :] + fcc).reshape(-1, 3)
    f = scaled(A)
    A = A[np.all((f >= 0) & (f < det), axis=1)]

    def key(x):
        """One integer per lattice point modulo the cell."""
        x = x - np.floor_divide(scaled(x), det) @ Q
        span = np.int64(8 * (int(np.abs(Q).sum()) + 8))
        return ((x[:, 0] + span) * (2 * span) + x[:, 1] + span) * (2 * span) + x[:, 2] + span

    keys = key(A)
    order = np.argsort(keys)
    signs = []
    for step in ((2, 0, 2), (2, 0, -2)):
        nxt = order[np.searchsorted(keys[order], key(A + np.array(step)))]
        label, jump = np.arange(len(A)), nxt
        for _ in range(int(math.ceil(math.log2(len(A)))) + 1):
            label = np.minimum(label, label[jump])
            jump = jump[jump]
        signs.append(rng.integers(0, 2, len(A))[label].astype(bool))
    d = np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1], [-1, -1, 1]])
    p, q = signs[0][:, None], signs[1][:, None]
    # an A site gives along d0 or d2 and along d1 or d3; the B site reached
    # from it along d0 lies on its first chain, the B site along d1 on the
    # second, so a B site takes its second sign from the A site at -d1
    a_dirs = np.stack([np.where(p, d[0], d[2]), np.where(q, d[1], d[3])], 1)
    B = A + d[0]
    q_b = signs[1][order[np.searchsorted(keys[order], key(B - d[1]))]][:, None]
    b_dirs = np.stack([np.where(p, -d[2], -d[0]), np.where(q_b, -d[3], -d[1])], 1)
    sites = np.concatenate([A, B]).astype(float)
    dirs = np.concatenate([a_dirs, b_dirs]).astype(float)
    frac = sites @ np.linalg.inv(Q.astype(float))
    return frac - np.floor(frac), dirs


@lru_cache(maxsize=None)
def _strand(n, seed):
    """A zigzag chain of n carbons with 0-3 hydrogens each: positions along z,
    and its parameters, bonded terms and exceptions, numbered from 0."""
    rng = np.random.default_rng([n, seed])
    half = math.radians(55.5)
    rise, amp = 0.153 * math.sin(half), 0.5 * 0.153 * math.cos(half)
    pos, group, mass, charge, sigma, eps, cons, bonds, heavy = [], [], [], [], [], [], [], [], []
    adjacent = []

    def add(p, g, m, q, s, e):
        pos.append(p)
        group.append(g)
        mass.append(m)
        charge.append(q)
        sigma.append(s)
        eps.append(e)
        adjacent.append(set())
        return len(pos) - 1

    ch = math.radians(54.75)
    for i in range(n):
        side = 1.0 if i % 2 == 0 else -1.0
        p = np.array([side * amp, 0.0, (i - 0.5 * (n - 1)) * rise])
        out = np.array([side * math.cos(ch), 0.0, 0.0])
        hs = [out + np.array([0, math.sin(ch), 0]), out - np.array([0, math.sin(ch), 0])]
        if i == 0:
            hs.append(np.array([-side * math.sin(half), 0, -math.sin(half)]))
        if i == n - 1:
            hs.append(np.array([-side * math.sin(half), 0, math.sin(half)]))
        hs = [h / np.linalg.norm(h) for h in hs]
        keep = len(hs) if 0 in (i, n - 1 - i) else int(rng.choice([0, 1, 1, 2, 2]))
        c = add(p, i, 12.011, 0.0, float(rng.uniform(0.30, 0.40)), float(rng.uniform(0.2, 0.9)))
        if heavy:
            bonds.append((heavy[-1], c))
            adjacent[heavy[-1]].add(c)
            adjacent[c].add(heavy[-1])
        heavy.append(c)
        for h in hs[:keep]:
            k = add(p + 0.109 * h, i, 1.008, float(rng.uniform(0.05, 0.2)), 0.2649, 0.0657)
            cons.append((c, k, 0.109))
            adjacent[c].add(k)
            adjacent[k].add(c)
    charge = np.array(charge) + np.where(np.array(mass) > 2, rng.normal(0, 0.15, len(mass)), 0.0)
    is_heavy = np.array(mass) > 2
    charge[is_heavy] -= charge.sum() / is_heavy.sum()
    x = np.array(pos)

    def length(i, j):
        return float(np.linalg.norm(x[i] - x[j]))

    bond = [(i, j, length(i, j), 259408.0) for i, j in bonds]
    angle, torsion, exceptions = [], [], []
    for j, near in enumerate(adjacent):
        near = sorted(near)
        for a in range(len(near)):
            for b in range(a + 1, len(near)):
                u, v = x[near[a]] - x[j], x[near[b]] - x[j]
                t = math.acos(max(-1.0, min(1.0, float(u @ v) / (np.linalg.norm(u) * np.linalg.norm(v)))))
                light = (mass[near[a]] < 2) + (mass[near[b]] < 2)
                angle.append((near[a], j, near[b], t, (418.4, 292.88, 276.14)[light]))
    for a, b, c, d in zip(heavy, heavy[1:], heavy[2:], heavy[3:]):
        torsion.append((a, b, c, d, int(rng.integers(1, 4)), float(rng.uniform(0, math.pi)), float(rng.uniform(0, 10))))
    for i in range(len(x)):
        one2 = adjacent[i]
        one3 = set().union(*[adjacent[j] for j in one2]) - {i} - one2
        one4 = set().union(*[adjacent[j] for j in one3]) - {i} - one2 - one3 if one3 else set()
        exceptions += [(i, j, 0.0, 1.0, 0.0) for j in sorted(one2 | one3) if j > i]
        exceptions += [(i, j, charge[i] * charge[j] / 1.2, 0.5 * (sigma[i] + sigma[j]), 0.5 * math.sqrt(eps[i] * eps[j]))
                       for j in sorted(one4) if j > i]
    return dict(pos=x, group=np.array(group), mass=np.array(mass), charge=charge, sigma=np.array(sigma),
                eps=np.array(eps), cons=cons, bond=bond, angle=angle, torsion=torsion, exc=exceptions,
                heavy=np.array(heavy))


def _smooth(n):
    while True:
        r = n
        for p in (2, 3, 5, 7):
            while r % p == 0:
                r //= p
        if r == 1:
            return n
        n += 1


def _alpha():
    return math.sqrt(-math.log(2 * TOLERANCE)) / CUTOFF


def _mesh(mesh, box):
    """mesh > 0: that many points per axis; 0: per axis, the smallest size the
    Ewald tolerance asks for with factors 2, 3, 5, 7; -1: a multiple of 8 at or
    above it, the same on every axis, 32-128."""
    least = [max(6, math.ceil(2 * _alpha() * box[k][k] / (3 * TOLERANCE ** 0.2))) for k in range(3)]
    if mesh > 0:
        return (mesh,) * 3
    if mesh < 0:
        n = min(128, max(32, 8 * math.ceil(max(least) / 8)))
        while _smooth(n) != n:
            n += 8
        return (n,) * 3
    return tuple(_smooth(n) for n in least)


@lru_cache(maxsize=64)
def _topology(shape, cells, mesh, restraint, barostat):
    """The system of one cell and what its coordinates are made from."""
    M = _cell(shape, cells)
    rng = np.random.default_rng([int(abs(np.linalg.det(M))), M.shape[0]])
    frac, dirs = _lattice(M)
    # the cell in OpenMM's lower-triangular orientation: the Cholesky factor of
    # the lattice vectors' products; directions turn with it
    L = np.linalg.cholesky((M @ M.T).astype(float))
    box = L * LATTICE
    turn = np.linalg.inv(M.astype(float)) @ L
    oxygen = frac @ box
    dirs = (dirs @ turn) / math.sqrt(3.0)
    volume = float(np.prod(np.diag(box)))
    faces = [np.linalg.norm(np.cross(box[(a + 1) % 3], box[(a + 2) % 3])) for a in range(3)]
    radius = 0.5 * volume / max(faces) - 0.35
    centre = 0.5 * box.sum(0)
    # strands on a square grid, innermost first, until a tenth of the atoms
    wanted = 0.1 * 3 * len(oxygen)
    spots = [(i * i + j * j, i, j) for i in range(-40, 41) for j in range(-40, 41)]
    strands, count = [], 0
    for r2, i, j in sorted(spots):
        length = 2 * math.sqrt(max(0.0, radius ** 2 - 0.48 ** 2 * r2))
        n = min(60, int((length - 0.2) / 0.1261))
        if n < 5 or count >= wanted:
            continue
        s = _strand(n, (i + 3 * j) % 4)
        strands.append((s, centre + 0.48 * np.array([i, j, 0.0])))
        count += len(s["mass"])
    solute = np.concatenate([s["pos"] + at for s, at in strands]) if strands else np.zeros((0, 3))
    # waters clear of the strands; a few left out at random, so that counts are
    # not round; the last of them ions
    keep = np.ones(len(oxygen), bool)
    if strands:
        keep = _clear(oxygen, solute, box, 0.30)
    keep = np.nonzero(keep)[0]
    keep = np.sort(rng.permutation(keep)[: len(keep) - 1 - len(keep) // 200])
    ions = 2 * max(1, len(keep) // 3300)
    ion_at = rng.choice(keep, ions, replace=False)
    water = np.setdiff1d(keep, ion_at)
    w = len(water)

    q_o, q_h, r_oh, r_hh = -0.834, 0.417, 0.09572, 0.15139
    up = dirs[water, 0] + dirs[water, 1]
    up /= np.linalg.norm(up, axis=1)[:, None]
    across = dirs[water, 0] - dirs[water, 1]
    across /= np.linalg.norm(across, axis=1)[:, None]
    half = 0.5 * r_hh
    height = math.sqrt(r_oh ** 2 - half ** 2)
    local = np.stack([np.zeros((w, 3)), height * up + half * across, height * up - half * across], 1)

    def cat(name, ion, waters):
        return np.concatenate([s[name] for s, _ in strands] + [np.asarray(ion, float), np.tile(waters, w)])

    na = np.arange(ions) % 2 == 0
    mass = cat("mass", np.where(na, 22.99, 35.453), [15.999, 1.008, 1.008])
    charge = cat("charge", np.where(na, 1.0, -1.0), [q_o, q_h, q_h])
    sigma = cat("sigma", np.where(na, 0.2439, 0.4478), [0.315075, 0.0, 0.0])
    eps = cat("eps", np.where(na, 0.3658, 0.1489), [0.635968, 0.0, 0.0])
    rows = {k: [] for k in ("cons", "bond", "angle", "torsion", "exc")}
    width = {"cons": (2, 3), "bond": (2, 4), "angle": (3, 5), "torsion": (4, 7), "exc": (2, 5)}
    group, heavy, start, groups = [], [], 0, 0
    for s, _ in strands:
        for k in rows:
            r = np.array(s[k], float).reshape(-1, width[k][1])
            r[:, : width[k][0]] += start
            rows[k].append(r)
        group.append(s["group"] + groups)
        heavy.append(s["heavy"] + start)
        groups += int(s["group"].max()) + 1
        start += len(s["mass"])
    first = start + ions + 3 * np.arange(w)
    o, h1, h2 = first, first + 1, first + 2
    one = np.ones(w)
    rows["cons"].append(np.concatenate([np.stack([o, h1, r_oh * one], 1), np.stack([o, h2, r_oh * one], 1),
                                        np.stack([h1, h2, r_hh * one], 1)]))
    rows["exc"].append(np.concatenate([np.stack([a, b, 0 * one, one, 0 * one], 1)
                                       for a, b in ((o, h1), (o, h2), (h1, h2))]))
    rows = {k: np.concatenate(v) if v else np.zeros((0, width[k][1])) for k, v in rows.items()}

    def col(k, c):
        return rows[k][:, c].astype(np.int32) if c < width[k][0] else rows[k][:, c].copy()

    box_rows = reduceBox(box)
    forces = [
        HarmonicBondForce(*[col("bond", c) for c in range(4)]),
        HarmonicAngleForce(*[col("angle", c) for c in range(5)]),
        PeriodicTorsionForce(*[col("torsion", c) for c in range(4)], col("torsion", 4).astype(np.int32),
                             col("torsion", 5), col("torsion", 6)),
        NonbondedForce(charge=charge, sigma=sigma, epsilon=eps, exceptionP1=col("exc", 0), exceptionP2=col("exc", 1),
                       exceptionChargeProd=col("exc", 2), exceptionSigma=col("exc", 3), exceptionEpsilon=col("exc", 4),
                       cutoff=CUTOFF, ewaldTolerance=TOLERANCE, grid=_mesh(mesh, box_rows),
                       useDispersionCorrection=True, recipForceGroup=1),
        CMMotionRemover(1),
    ]
    if restraint and strands:
        hv = np.concatenate(heavy).astype(np.int32)
        forces.append(PositionRestraintForce(hv, np.full(len(hv), restraint), solute[hv, 0].copy(),
                                             solute[hv, 1].copy(), solute[hv, 2].copy()))
    if barostat:
        forces.append(MonteCarloBarostat(1.0, TEMPERATURE, barostat, 1))
    system = OpenMMSystem(boxVectors=tuple(tuple(float(v) for v in r) for r in box_rows), masses=mass,
                          constraintP1=col("cons", 0), constraintP2=col("cons", 1), constraintDistance=col("cons", 2),
                          forces=forces)
    return dict(system=system, solute=solute, group=np.concatenate(group) if group else np.zeros(0, int),
                groups=groups, ions=oxygen[ion_at], oxygen=oxygen[water], local=local, volume=volume)


def _clear(sites, solute, box, limit):
    """Which sites keep `limit` from every solute atom: the solute binned into
    cells of that width, each site looking at the 27 around it (the strands
    stay inside the cell, so no images are needed)."""
    lo = solute.min(0) - 2 * limit
    n = (np.ceil((solute.max(0) - lo) / limit) + 3).astype(int)
    grid = {}
    for k, c in enumerate(map(tuple, ((solute - lo) / limit).astype(int))):
        grid.setdefault(c, []).append(k)
    near = np.zeros(n, bool)
    for c in grid:
        near[c[0] - 1:c[0] + 2, c[1] - 1:c[1] + 2, c[2] - 1:c[2] + 2] = True
    keep = np.ones(len(sites), bool)
    for image in np.stack(np.meshgrid([-1, 0, 1], [-1, 0, 1], [-1, 0, 1], indexing="ij"), -1).reshape(-1, 3) @ box:
        x = sites + image
        cell = np.floor((x - lo) / limit).astype(int)
        ok = np.all((cell >= 1) & (cell < n - 1), axis=1)
        for k in np.nonzero(ok)[0][near[tuple(cell[ok].T)]]:
            c = cell[k]
            js = [j for dx in (-1, 0, 1) for dy in (-1, 0, 1) for dz in (-1, 0, 1)
                  for j in grid.get((c[0] + dx, c[1] + dy, c[2] + dz), ())]
            if js and np.min(np.sum((solute[js] - x[k]) ** 2, axis=1)) < limit ** 2:
                keep[k] = False
    return keep


def _coordinates(top, rng):
    """Thermally displaced positions and Maxwell-Boltzmann velocities, (N, 3).
    The velocities are drawn cool: the displaced lattice gives up potential
    energy in the first steps, which brings the temperature to about 300 K."""
    w = len(top["oxygen"])
    solute = top["solute"] + rng.normal(0, 0.002, (top["groups"], 3))[top["group"]] if top["groups"] else top["solute"]
    # a small rotation vector per water (Rodrigues' formula)
    r = rng.normal(0, 0.12, (w, 3))
    a = np.linalg.norm(r, axis=1)[:, None, None]
    k = (r / a[:, 0])[:, None, :]
    v = top["local"]
    turned = v * np.cos(a) + np.cross(k, v) * np.sin(a) + k * np.sum(k * v, -1, keepdims=True) * (1 - np.cos(a))
    water = (top["oxygen"] + rng.normal(0, 0.008, (w, 3)))[:, None, :] + turned
    x = np.concatenate([solute, top["ions"] + rng.normal(0, 0.008, top["ions"].shape), water.reshape(-1, 3)])
    m = top["system"].masses[:, None]
    u = np.sqrt(KB * 0.5 * TEMPERATURE / m) * rng.normal(0, 1, x.shape)
    return x, u - (m * u).sum(0) / m.sum()


# ---- one pass ---------------------------------------------------------------------

def _network():
    """The warm-start network's weights as a user's file holds them: SHAKE's
    first-order update, multiplier = 100 (d^2 - |r'|^2) / d^2, carried through
    the hidden layers in their linear range (weights are powers of two)."""
    w1, w2, w3 = np.zeros((32, 64)), np.zeros((64, 64)), np.zeros((64, 16))
    for c in range(4):
        w1[4 * c, c] = 2.0 ** -7
        w2[c, c] = 1.0
        w3[c, c] = 2.0 ** 7
    return np.concatenate([p.reshape(-1) for p in (w1, np.zeros(64), w2, np.zeros(64), w3, np.zeros(16))])


def prepare(case, seed):
    rng = np.random.default_rng([int(seed), 71])
    engines = []
    for k, top in enumerate(_systems(case)):
        x, v = _coordinates(top, rng)
        system = top["system"]
        engines.append(HipEngine(system, OpenMMState(system.boxVectors, x.reshape(-1), v.reshape(-1)),
                                 RunOptions(timeStep=DT, temperature=TEMPERATURE, friction=1.0,
                                            constraintTolerance=1e-6, seed=int(seed) * 64 + k,
                                            integrator="Verlet" if case.get("verlet") else "LangevinMiddle")))
    state = {"case": case, "engines": engines}
    if case["job"] in ("forces", "minimise"):
        state["positions"] = x.reshape(-1)
    if case["job"] == "batch":
        if case.get("learned"):
            state["network"] = native.NativeWarmStart()
            state["network"].set_params(_network())
            for e in engines:
                state["network"].attach(e._native)
        state["batch"] = HipBatch(engines)
    return state


def run(state):
    case, engines = state["case"], state["engines"]
    if case["job"] == "forces":
        energy, forces = engines[0].potential(state["positions"])
        return {"energy": np.float32(energy), "forces": forces.astype(np.float32)}
    if case["job"] == "minimise":
        engines[0].setPositions(state["positions"])
        engines[0].minimise(case["iterations"], 1.0)
        return {"positions": engines[0].positions().astype(np.float32)}
    if case["job"] == "batch":
        state["batch"].run(case["steps"])
        return {"positions": np.concatenate([e.positions() for e in engines]).astype(np.float32),
                "velocities": np.concatenate([e.velocities() for e in engines]).astype(np.float32)}
    e = engines[0]
    e.run(case["steps"])
    out = {"positions": e.positions().astype(np.float32), "velocities": e.velocities().astype(np.float32)}
    if case.get("barostat"):
        out["box"] = np.array(e.boxVectors(), dtype=np.float32)
    return out


def work(case):
    """Per step: 76 flops per in-cutoff pair, the mesh transforms (5 n log2 n
    each way over a real grid, both ways) and 125 points per charge spread and
    gathered; positions, velocities, the integrator's residual and the mesh
    read and written once."""
    steps = {"run": case.get("steps", 1), "batch": case.get("steps", 1), "forces": 1,
             "minimise": case.get("iterations", 1)}[case["job"]]
    flops = bytes_ = 0.0
    for top in _systems(case):
        n = top["system"].particleCount
        mesh = np.array(top["system"].force("NonbondedForce").grid, float)
        points = float(mesh.prod())
        pairs = 0.5 * n * n / top["volume"] * 4 / 3 * math.pi * CUTOFF ** 3
        flops += 76 * pairs + 5 * points * math.log2(points) + 125 * n * 12
        bytes_ += 124 * n + 16 * points
    return {"bytes": steps * bytes_, "flops": steps * flops}


# ---- the same forces in 64 bits -------------------------------------------------------

def exact(case, seed):
    if case["job"] != "forces":
        return None
    top = _systems(case)[0]
    # the coordinates prepare() draws, on the engine's 2^-32 nm grid
    x, _ = _coordinates(top, np.random.default_rng([int(seed), 71]))
    device = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.tensor(np.rint(x * 2.0 ** 32) * 2.0 ** -32, device=device)
    energy, forces = _potential(top["system"], x)
    return {"energy": energy, "forces": forces.reshape(-1).cpu().numpy()}


def _potential(system, x):
    """Energy and forces of every term in float64: forces by differentiation."""
    n, device = x.shape[0], x.device
    alpha = _alpha()
    box = torch.tensor(system.boxVectors, dtype=torch.float64, device=device)

    def on(a):
        return torch.as_tensor(np.asarray(a), device=device)

    def images(d):
        for k in (2, 1, 0):
            d = d - torch.floor(d[:, k:k + 1] / box[k, k] + 0.5) * box[k]
        return d

    nb = system.force("NonbondedForce")
    q, sig, eps = on(nb.charge), on(nb.sigma), on(nb.epsilon)
    p1, p2 = on(nb.exceptionP1).long(), on(nb.exceptionP2).long()
    excluded = torch.unique(torch.minimum(p1, p2) * n + torch.maximum(p1, p2))
    grad = torch.zeros_like(x)
    total = 0.0

    def add(energy, at):
        """Accumulates an energy that depends on the leaf `at`."""
        nonlocal total, grad
        total += float(energy.detach())
        grad += torch.autograd.grad(energy, at)[0]

    # direct space, a block of rows at a time
    rows = max(1, int(4e7) // n)
    for a in range(0, n, rows):
        i = torch.arange(a, min(n, a + rows), device=device)
        d = images((x[None, a:] - x[i, None]).reshape(-1, 3))
        hit = torch.nonzero((d * d).sum(1) < CUTOFF ** 2).reshape(-1)
        pi, pj = i[hit // (n - a)], a + hit % (n - a)
        ok = pj > pi
        pi, pj = pi[ok], pj[ok]
        ok = ~torch.isin(pi * n + pj, excluded)
        pi, pj = pi[ok], pj[ok]
        del d
        y = x.clone().requires_grad_(True)
        r = images(y[pj] - y[pi]).norm(dim=1)
        s6 = ((0.5 * (sig[pi] + sig[pj])) / r) ** 6
        lj = 4 * torch.sqrt(eps[pi] * eps[pj]) * (s6 * s6 - s6)
        add((COULOMB * q[pi] * q[pj] * torch.erfc(alpha * r) / r + lj).sum(), y)
    y = x.clone().requires_grad_(True)
    # exclusions and exceptions
    r = images(y[p2] - y[p1]).norm(dim=1)
    s6 = (on(nb.exceptionSigma) / r) ** 6
    e = (COULOMB * (on(nb.exceptionChargeProd) - q[p1] * q[p2] * torch.erf(alpha * r)) / r
         + 4 * on(nb.exceptionEpsilon) * (s6 * s6 - s6)).sum()
    # bonds, angles, torsions, restraints
    f = system.force("HarmonicBondForce")
    e = e + (0.5 * on(f.k) * ((y[on(f.p2).long()] - y[on(f.p1).long()]).norm(dim=1) - on(f.length)) ** 2).sum()
    f = system.force("HarmonicAngleForce")
    u, v = (y[on(p).long()] - y[on(f.p2).long()] for p in (f.p1, f.p3))
    angle = torch.atan2(torch.linalg.cross(u, v).norm(dim=1), (u * v).sum(1))
    e = e + (0.5 * on(f.k) * (angle - on(f.angle)) ** 2).sum()
    f = system.force("PeriodicTorsionForce")
    a, b, c, d = (y[on(p).long()] for p in (f.p1, f.p2, f.p3, f.p4))
    b1, b2, b3 = b - a, c - b, d - c
    n1, n2 = torch.linalg.cross(b1, b2), torch.linalg.cross(b2, b3)
    phi = torch.atan2(b2.norm(dim=1) * (b1 * n2).sum(1), (n1 * n2).sum(1))
    e = e + (on(f.k) * (1 + torch.cos(on(f.periodicity) * phi - on(f.phase)))).sum()
    f = system.force("PositionRestraint")
    if f is not None:
        ref = torch.stack([on(f.x0), on(f.y0), on(f.z0)], 1)
        e = e + (on(f.k) * (images(y[on(f.particle).long()] - ref) ** 2).sum(1)).sum()
    # the mesh: order-5 B-splines, the grid's transform, the Ewald factor
    mesh = [int(g) for g in nb.grid]
    u = (y @ torch.linalg.inv(box)) * torch.tensor(mesh, dtype=torch.float64, device=device)
    cell = torch.floor(u.detach())
    w = u - cell
    theta = [torch.stack([1 - w, w])]  # order 2, then up to order 5
    for order in (3, 4, 5):
        t = theta[-1]
        zero = torch.zeros_like(t[:1])
        k = torch.arange(order, device=device, dtype=torch.float64)[:, None, None]
        # spline j of this order at w is M(w + order - 1 - j)
        z = w[None] + (order - 1 - k)
        theta.append((z * torch.cat([zero, t]) + (order - z) * torch.cat([t, zero])) / (order - 1))
    t = theta[-1]
    at = [(cell[:, k, None].long() - 4 + torch.arange(5, device=device)) % mesh[k] for k in range(3)]
    index = (at[0][:, :, None, None] * mesh[1] + at[1][:, None, :, None]) * mesh[2] + at[2][:, None, None, :]
    # theta[j] weighs the point floor(u) - 4 + j
    value = (q[:, None, None, None] * t[:, :, 0].T[:, :, None, None] * t[:, :, 1].T[:, None, :, None]
             * t[:, :, 2].T[:, None, None, :])
    grid = torch.zeros(mesh[0] * mesh[1] * mesh[2], dtype=torch.float64, device=device)
    grid = grid.index_add(0, index.reshape(-1), value.reshape(-1)).reshape(mesh)
    knots = np.array([1, 11, 11, 1]) / 24.0
    mod = []
    for g in mesh:
        m = np.abs(np.exp(2j * np.pi * np.outer(np.arange(g), np.arange(4)) / g) @ knots) ** 2
        low = np.nonzero(m < 1e-7)[0]
        m[low] = 0.5 * (m[low - 1] + m[(low + 1) % g])
        mod.append(torch.tensor(m, device=device))
    freq = [torch.fft.fftfreq(g, 1.0 / g, dtype=torch.float64, device=device) for g in mesh]
    m = torch.stack(torch.meshgrid(*freq, indexing="ij"), -1)
    k2 = ((m @ torch.linalg.inv(box).T) ** 2).sum(-1) * (2 * math.pi) ** 2
    k2[0, 0, 0] = 1.0
    volume = float(torch.linalg.det(box))
    factor = 2 * math.pi * COULOMB / volume * torch.exp(-k2 / (4 * alpha ** 2)) / (
        k2 * mod[0][:, None, None] * mod[1][None, :, None] * mod[2][None, None, :])
    factor[0, 0, 0] = 0.0
    e = e + (factor * torch.fft.fftn(grid).abs() ** 2).sum()
    add(e, y)
    # self energy, net charge, and the dispersion tail over all pairs (i <= j)
    total += -COULOMB * alpha / math.sqrt(math.pi) * float((q * q).sum())
    total += -math.pi * COULOMB * float(q.sum()) ** 2 / (2 * alpha ** 2 * volume)
    kinds, count = np.unique(np.stack([nb.sigma, nb.epsilon], 1), axis=0, return_counts=True)
    s = 0.5 * (kinds[:, None, 0] + kinds[None, :, 0])
    ep = np.sqrt(kinds[:, None, 1] * kinds[None, :, 1])
    times = 0.5 * (np.outer(count, count) + np.diag(count))
    pairs = 0.5 * n * (n + 1.0)
    total += 8 * math.pi * n * float(n) / volume * float(
        (times * ep * s ** 12).sum() / pairs / (9 * CUTOFF ** 9) - (times * ep * s ** 6).sum() / pairs / (3 * CUTOFF ** 3))
    return total, -grad
