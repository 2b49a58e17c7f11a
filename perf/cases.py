"""The framework's measured workloads: whole solves of input decks and batched ensembles.

A pass is what a user's program does with one deck or one batch of decks through the public entry
points: build the solver, run the cellular automaton to its termination check (or to a given
cycle, or one time step at a time), and read the fields back. Decks are written by ``prepare``; the
random-stream seed of a solve comes from the case's seed, so another seed is another substrate and
other nuclei. Every size and option is one of the repository's example decks, of its tests' or
benchmark's workloads, or of the same generic family.

Outputs are the fields and counters a program reads after a solve. They are whole numbers
(cell types, grain indices, counts), with two exceptions that have no closed form: the
half-diagonals of a solve that is stopped mid-run, and the means of the grain statistics.
"""
from __future__ import annotations

import math
import random
import tempfile
from pathlib import Path

import numpy as np

import exaca_amd as ea
from exaca_amd import decks

# Bytes a cell cannot do without over its life: one frontier evaluation (137: its state and the 26
# critical lengths), its capture (125: the new octahedron), its solidification (1) and the two
# fields read back (8). Flops of its capture: 26 critical lengths of 4 faces and the octahedron.
CELL_BYTES = 137 + 125 + 1 + 8
CELL_FLOPS = 1200


def _c(name, nx, ny, nz, **k):
    case = dict(name=name, kind="directional", nx=nx, ny=ny, nz=nz, G=1e6, R=1e6, N=10, density=10.0,
                fraction=0.04, cycles=0, drive="run", stats=False)
    case.update(k)
    return case


def _s(name, nsx, nsy, offset, radius, **k):
    case = dict(name=name, kind="spots", nsx=nsx, nsy=nsy, offset=offset, radius=radius, G=1e6, R=1e6, N=10,
                density=10.0, spacing=25, layers=1, layer_height=20)
    case.update(k)
    return case


def _e(name, count, side_min, side_max, mix):
    return dict(name=name, kind="ensemble", count=count, side_min=side_min, side_max=side_max, mix=mix)


def listed():
    return [
        # the smallest solve in use (the smoke test's): every step is latency
        _c("directional_24", 24, 24, 24),
        # odd sides, many nuclei: no dimension a multiple of anything
        _c("directional_37x23x31", 37, 23, 31, density=200.0, fraction=0.1),
        # a program that calls the time-step functions itself, one Nucleation and one CellCapture
        # per cycle and a check at the end, as the reference's loop does
        _c("stepwise_48", 48, 48, 48, density=400.0, fraction=0.02, cycles=400, drive="step"),
        # the small example deck: substrate grains only, fine time step
        _c("directional_50_substrate", 50, 50, 50, G=5e5, R=3e5, N=25, density=0.0, fraction=0.005),
        # the baseline deck of 100^3 with its grain statistics
        _c("directional_100_stats", 100, 100, 100, stats=True),
        # the largest process-map side
        _c("directional_256", 256, 256, 256),
        # the large single-domain solve
        _c("directional_400", 400, 400, 400),
        # the benchmark's full width over its bottom planes, stopped mid-run: the widest front
        _c("directional_800x800x40_mid", 800, 800, 40, cycles=1000),
        # the small spot-melt example: two overlapping spots, a fine time step, many quiet cycles
        _s("spots_1x2_example", 1, 2, 25, 25, G=5e5, R=3e5, N=25),
        # several layers of overlapping spots with dense nuclei: layer transitions and remelted rims
        _s("spots_2x2_two_layers", 2, 2, 16, 10, density=300.0, spacing=8, layers=2, layer_height=6),
        # a process map of small domains, all resident at once
        _e("ensemble_64_small", 64, 32, 64, 2024),
        # fewer, larger domains of the process map
        _e("ensemble_16_large", 16, 64, 192, 2024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("cube", "box", "box", "wide", "step", "spots", "ensemble"))
    if kind == "cube":
        n = _log_int(rng, 16, 256)
        c = _c("", n, n, n, density=float(_log_int(rng, 1, 400)), fraction=round(rng.uniform(0.01, 0.1), 3),
               stats=rng.random() < 0.5)
    elif kind == "box":
        c = _c("", _log_int(rng, 12, 256), _log_int(rng, 12, 256), _log_int(rng, 12, 160),
               density=float(_log_int(rng, 1, 400)), fraction=round(rng.uniform(0.005, 0.2), 3),
               G=float(_log_int(rng, 500000, 2000000)))
    elif kind == "wide":
        c = _c("", _log_int(rng, 300, 800), _log_int(rng, 300, 800), _log_int(rng, 16, 48),
               cycles=rng.randrange(200, 1001))
    elif kind == "step":
        c = _c("", _log_int(rng, 16, 96), _log_int(rng, 16, 96), _log_int(rng, 16, 96), density=100.0,
               cycles=rng.randrange(100, 801), drive="step")
    elif kind == "spots":
        c = _s("", rng.randrange(1, 3), rng.randrange(1, 3), rng.randrange(12, 31), rng.randrange(12, 23),
               density=float(_log_int(rng, 10, 300)), spacing=rng.randrange(6, 13), layers=rng.randrange(1, 3),
               layer_height=rng.randrange(4, 9))
    else:
        lo = rng.randrange(20, 49)
        c = _e("", rng.randrange(4, 41), lo, lo * 2 + rng.randrange(0, 33), rng.randrange(1 << 20))
    del c["name"]
    return c


_SPOT_DECK = """spot melt array
*****
Problem type: S
Decomposition strategy (1 for 1D domain decomposition, 2 for simple 2D decomposition, 3 for complex 2D decomposition): 1
Material: Inconel625_Baseline
Cell size (microns): 1
Heterogeneous nucleation density (normalized by 1*10^12 per m^3): {density}
Mean nucleation undercooling (in K): 5
Standard deviation of nucleation undercooling: 0.5
Path to output: ./
Output file base name: spots
File of grain orientations: GrainOrientationVectors_Robert.csv
Thermal gradient (K/m): {G}
Cooling rate (K/s): {R}
Number of spots in x: {nsx}
Number of spots in y: {nsy}
Offset between spot centers (in microns): {offset}
Radii of spots (in microns): {radius}
Number of layers: {layers}
Offset between layers (in cells): {layer_height}
"N", where the time step = deltax/(Steady State Velocity * N): {N}
Substrate grain spacing (in microns): {spacing}
***Output data printing options: (Y or N) which data should be printed***
Print Paraview vtk file of grain misorientation values (Y or N)?: N
Print Paraview vtk file of all ExaCA data for post-processing (Y or N)?: N
Debug check (reduced)- Print data for main Kokkos views (CellType, LayerID, CritTimeStep) following initialization for debug check (Y or N)?: N
Debug check (extensive) - Print data for all main data structures (CellType, GrainID, CritTimeStep, UndercoolingCurrent, UndercoolingChange, Melted, LayerID) following initialization for debug check (Y or N)?: N
"""


def _mix(case):
    """Sides, thermal gradient, cooling rate and nucleation density of an ensemble's domains."""
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["count"]):
        sides = [_log_int(r, case["side_min"], case["side_max"]) for _ in range(3)]
        G = math.exp(r.uniform(math.log(3e5), math.log(1e7)))
        R = math.exp(r.uniform(math.log(1e4), math.log(1e7)))
        density = math.exp(r.uniform(math.log(0.1), math.log(100.0)))
        out.append((*sides, G, R, density))
    return out


class _Batch:
    """An ensemble handle kept by the program, and its host-initialised domains."""

    def __init__(self, prepared):
        self.prepared = prepared
        need = sum(p.device_bytes for p in prepared)
        self.ensemble = ea.Ensemble(len(prepared), need + (len(prepared) << 12))
        self.ensemble.set_blocks(32)

    def __del__(self):
        self.ensemble.close()
        for p in self.prepared:
            p.close()


def prepare(case, seed):
    where = tempfile.TemporaryDirectory(prefix="exaca_case_")
    path = Path(where.name) / "deck.txt"
    state = {"case": case, "seed": seed + 1, "where": where, "deck": path}
    if case["kind"] == "directional":
        decks.directional_deck(path, case["nx"], case["ny"], case["nz"], G=case["G"], R=case["R"], N=case["N"],
                               density=case["density"], fraction=case["fraction"])
    elif case["kind"] == "spots":
        path.write_text(_SPOT_DECK.format(**case))
    else:
        prepared = []
        for i, (nx, ny, nz, G, R, density) in enumerate(_mix(case)):
            decks.directional_deck(path, nx, ny, nz, G=G, R=R, density=density)
            prepared.append(ea.Prepared(path, seed + 1 + 7919 * i))
        state["batch"] = _Batch(prepared)
    return state


def _counters(sol):
    q = sol.query()
    return [q["nn"], q["frontier"], q["captures"], q["solidified"]]


def _solve(state):
    case = state["case"]
    with ea.Solver(state["deck"], seed=state["seed"]) as sol:
        out = {}
        cycles = case.get("cycles", 0)
        if case.get("drive") == "step":
            for cycle in range(1, cycles + 1):
                sol.step(cycle)
            out["cycle"], out["check"], _ = sol.check(cycles)
        else:
            out["cycle"], _ = sol.run(max_cycles=cycles)
        out["CellType"] = sol.field(ea.FIELD_CELLTYPE)
        out["GrainID"] = sol.field(ea.FIELD_GRAINID)
        if cycles:
            out["DiagonalLength"] = sol.field(ea.FIELD_DIAGONAL)
        if case.get("stats"):
            out["stats"] = sol.grain_stats()
            out["stats"]["histogram"] = np.array(out["stats"]["histogram"])
        out["counters"] = _counters(sol)
    return out


def _solve_batch(state):
    batch = state["batch"]
    ens = batch.ensemble
    slots = [ens.admit(p) for p in batch.prepared]
    while True:
        ens.advance(250)
        final, errors = ens.poll_errors()
        if all(final[s] > 0 for s in slots):
            break
    out = {"cycles": final, "errors": errors, "CellType": [], "GrainID": [], "counters": []}
    for s, p in zip(slots, batch.prepared):
        out["CellType"].append(ens.field(s, ea.FIELD_CELLTYPE, p.cells))
        out["GrainID"].append(ens.field(s, ea.FIELD_GRAINID, p.cells))
        q = ens.query(s)
        out["counters"].append([q["nn"], q["frontier"], q["captures"], q["solidified"]])
        ens.release(s)
    for key in ("CellType", "GrainID"):
        out[key] = np.concatenate(out[key])
    out["counters"] = np.array(out["counters"])
    return out


def run(state):
    return _solve_batch(state) if state["case"]["kind"] == "ensemble" else _solve(state)


def _cells(case):
    if case["kind"] == "directional":
        return case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "ensemble":
        return sum(nx * ny * nz for nx, ny, nz, *_ in _mix(case))
    # the melted half ellipsoids of the spots, at most the box that holds them, per layer
    r, o = case["radius"], case["offset"]
    box = ((case["nsx"] - 1) * o + 2 * r) * ((case["nsy"] - 1) * o + 2 * r) * r
    melt = case["nsx"] * case["nsy"] * (2.0 / 3.0) * math.pi * r ** 3
    first = min(box, melt)
    return int(first * (1 + (case["layers"] - 1) * min(1.0, case["layer_height"] / r)))


def _fraction_done(case):
    """The share of a directional domain that a run of `cycles` steps has solidified: the front
    needs about 10 steps per plane after its first few hundred."""
    if not case.get("cycles"):
        return 1.0
    return min(1.0, max(0.02, (case["cycles"] - 300) / (12.0 * case["nz"])))


def work(case):
    cells = _cells(case) * _fraction_done(case)
    return {"bytes": cells * CELL_BYTES, "flops": cells * CELL_FLOPS}


def exact(case, seed):
    return None  # a cellular automaton's fields: whole numbers, compared value by value
