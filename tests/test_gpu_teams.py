"""GPU: the kernel that runs many steps of a domain in one launch, at the cross-sections where the
number of its workgroups changes (the last of a size and the first of the next, to the first domain
that takes two launches a step), against the oracle, cell for cell. One workgroup also gets a
bottom plane full of grains, whose claimants exceed what it stages in LDS. Each domain is run three
ways: in one call, in calls of odd lengths (each settles and books its own last step), and through
the time-step functions with their check."""
import numpy as np
import pytest

import exaca_amd as ea
import oracle as orc
from conftest import DATA, c_deck

pytestmark = pytest.mark.gpu

CASES = {
    "46x46x9_full": dict(n=9, nx=46, ny=46, density=2000, fraction=1.0),
    "46x46x9": dict(n=9, nx=46, ny=46, density=2000, fraction=0.05),
    "47x47x9": dict(n=9, nx=47, ny=47, density=2000, fraction=0.05),
    "78x78x7": dict(n=7, nx=78, ny=78, density=1000, fraction=0.05),
    "79x79x7": dict(n=7, nx=79, ny=79, density=1000, fraction=0.05),
    "126x126x5": dict(n=5, nx=126, ny=126, density=500, fraction=0.05),
    "127x127x5": dict(n=5, nx=127, ny=127, density=500, fraction=0.05),
    "238x238x4": dict(n=4, nx=238, ny=238, density=200, fraction=0.05),
    "239x239x4": dict(n=4, nx=239, ny=239, density=200, fraction=0.05),
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
