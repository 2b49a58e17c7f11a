"""GPU: more due cells, claimants and captures in a step than a workgroup's LDS stages hold (due cells: 1024 with
two launches a step, 2048 in a team; captures of a round: 256 and 512 threads). By counting: where the step's
due cells or captures outnumber what the stages of all workgroups hold together, one of them takes several
rounds. Each case asserts the count, and equals the oracle."""
import numpy as np
import pytest

import exaca_amd as ea
import oracle as orc
from conftest import DATA, c_deck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,blocks,due,captures", [(196, 8, 8 * 1024, 8 * 256), (100, None, 2048, 512)])
def test_steps_beyond_the_stages_match_the_oracle(tmp_path, monkeypatch, side, blocks, due, captures):
    """blocks: two launches a step by that many workgroups; None: one workgroup of a team, left alone with the
    domain."""
    if blocks:
        monkeypatch.setenv("EXACA_BLOCKS", str(blocks))
    else:
        monkeypatch.setenv("EXACA_MEET_US", "0")
    deck = c_deck(tmp_path / "d.txt", 8, nx=side, ny=side, density=1000, fraction=1.0, N=1)
    osim = orc.OracleSim(deck, DATA)
    steps, before, most = 160, 0, 0
    for cycle in range(1, steps + 1):
        osim.step(cycle)
        now = osim.dims()["captures"]
        most, before = max(most, now - before), now
    print(f"[rounds] {side}: {most} captures in a step", flush=True)
    assert most > captures
    with ea.Solver(deck) as sol:
        assert sol.query()["list_len"] > due  # of the first step
        team = sol.team()["workgroups"]
        sol.run(max_cycles=steps)
        if blocks:
            assert team == 0
        else:
            assert team > 1 and sol.team()["alone"] == sol.team()["launches"] == 1
        q, d = sol.query(), osim.dims()
        for key in ("nn", "captures", "solidified", "frontier"):
            assert q[key] == d[key], (key, q[key], d[key])
        ct = sol.field(ea.FIELD_CELLTYPE)
        assert np.array_equal(ct, osim.field(orc.CELLTYPE))
        assert np.array_equal(sol.field(ea.FIELD_GRAINID), osim.field(orc.GRAINID))
        act = np.flatnonzero(ct == 2)
        assert np.array_equal(sol.field(ea.FIELD_DIAGONAL)[act], osim.field(orc.DIAGLEN)[act])
