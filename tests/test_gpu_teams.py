"""GPU: the kernel that runs many steps of a domain in one launch, at the cross-sections where the
number of its workgroups changes (the last of a size and the first of the next, to the first domains
that take two launches a step), against the oracle, cell for cell. One workgroup also gets a
domain where a third of the cells are nuclei: about 740 captures a step, more claimants than it
stages in LDS. Each domain is run three
ways: in one call, in calls of odd lengths (each settles and books its own last step), and through
the time-step functions with their check."""
import numpy as np
import pytest

import exaca_amd as ea
import oracle as orc
from conftest import DATA, c_deck

pytestmark = pytest.mark.gpu

CASES = {
    "32x32x9_full": dict(n=9, nx=32, ny=32, density=2000, fraction=1.0),
    "32x32x60_third_nuclei": dict(n=60, nx=32, ny=32, density=300000, fraction=1.0, N=1, G=1e5),
    "32x32x9": dict(n=9, nx=32, ny=32, density=2000, fraction=0.05),
    "33x33x9": dict(n=9, nx=33, ny=33, density=2000, fraction=0.05),
    "58x58x7_full": dict(n=7, nx=58, ny=58, density=1000, fraction=1.0),
    "59x59x7": dict(n=7, nx=59, ny=59, density=1000, fraction=0.05),
    "82x82x5": dict(n=5, nx=82, ny=82, density=1000, fraction=0.05),
    "83x83x5": dict(n=5, nx=83, ny=83, density=500, fraction=0.05),
    "138x138x4": dict(n=4, nx=138, ny=138, density=500, fraction=0.05),
    "139x139x4": dict(n=4, nx=139, ny=139, density=500, fraction=0.05),
    "148x148x4": dict(n=4, nx=148, ny=148, density=500, fraction=0.05),
    "149x149x4": dict(n=4, nx=149, ny=149, density=200, fraction=0.05),
    "188x188x4": dict(n=4, nx=188, ny=188, density=200, fraction=0.05),
    "189x189x4": dict(n=4, nx=189, ny=189, density=200, fraction=0.05),
}


def _same(sol, osim, tag):
    q, d = sol.query(), osim.dims()
    for key in ("nn", "captures", "solidified", "frontier"):
        assert q[key] == d[key], (tag, key, q[key], d[key])
    ct = sol.field(ea.FIELD_CELLTYPE)
    assert np.array_equal(ct, osim.field(orc.CELLTYPE)), f"{tag}: CellType"
    assert np.array_equal(sol.field(ea.FIELD_GRAINID), osim.field(orc.GRAINID)), f"{tag}: GrainID"
    act = ct == 2
    assert np.array_equal(sol.field(ea.FIELD_DIAGONAL)[act], osim.field(orc.DIAGLEN)[np.flatnonzero(act)]), f"{tag}: DiagonalLength"


@pytest.mark.parametrize("case", list(CASES))
def test_steps_in_one_launch_match_the_oracle(tmp_path, case):
    k = dict(CASES[case])
    deck = c_deck(tmp_path / "d.txt", k.pop("n"), **k)
    cycles = 420  # mid-run: active cells of every kind
    osim = orc.OracleSim(deck, DATA)
    osim.run(max_cycles=cycles)
    print(f"[teams] {case}", flush=True)
    with ea.Solver(deck) as sol:
        sol.run(max_cycles=cycles)
        _same(sol, osim, "one call")
        final = sol.run()[0]
    with ea.Solver(deck) as sol:
        for c in (1, 2, 5, 68, 131, 132, 401, cycles):
            sol.run(max_cycles=c)
        _same(sol, osim, "calls of odd lengths")
    with ea.Solver(deck) as sol:
        for c in range(1, cycles + 1):
            sol.step(c)
            if c % 140 == 0:
                sol.check(c)
        _same(sol, osim, "time-step functions")
    ocycle, _ = osim.run()
    assert final == ocycle
