"""GPU: EXACA_CAND_STAGE narrows the LDS stage of a team's claimants, so that most of them take the lists in
memory; values it never took are refused."""
import numpy as np
import pytest

import exaca_amd as ea
import oracle as orc
from conftest import DATA, c_deck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", ["0", "-3", "2049", "x"])
def test_bad_stages_are_refused(tmp_path, monkeypatch, bad):
    deck = c_deck(tmp_path / "d.txt", 8)
    prep = ea.Prepared(deck)
    with ea.Ensemble(1, prep.device_bytes + (1 << 16)) as ens:
        monkeypatch.setenv("EXACA_CAND_STAGE", bad)
        with pytest.raises(ea.ExacaError, match="EXACA_CAND_STAGE must be"):
            ea.Solver(deck)
        with pytest.raises(ea.ExacaError, match="EXACA_CAND_STAGE must be"):
            ens.admit(prep)
        monkeypatch.delenv("EXACA_CAND_STAGE")
        assert ens.admit(prep) == 0  # the refused one took neither slot nor memory


CASES = [
    (dict(n=24, nx=20, ny=20, density=3000, fraction=0.1), 1, 1),
    (dict(n=16, nx=44, ny=44, density=2000, fraction=0.1), 2, 8),
    # a quarter of the cells nuclei: hundreds of claimants a step
    (dict(n=60, nx=30, ny=30, density=300000, fraction=1.0, N=1, G=1e5), 16, 32),
]


@pytest.mark.parametrize("deck,stage,workgroups", CASES)
def test_claimants_beyond_the_stage_match_the_oracle(tmp_path, monkeypatch, deck, stage, workgroups):
    monkeypatch.setenv("EXACA_CAND_STAGE", str(stage))
    k = dict(deck)
    path = c_deck(tmp_path / "d.txt", k.pop("n"), **k)
    osim = orc.OracleSim(path, DATA)
    osim.run(max_cycles=420)
    with ea.Solver(path) as sol:
        sol.run(max_cycles=420)
        team, q, d = sol.team(), sol.query(), osim.dims()
        print(f"[stage] {stage}: {team}", flush=True)
        assert team["workgroups"] == workgroups and team["spilled"] > 0
        for key in ("nn", "captures", "solidified", "frontier"):
            assert q[key] == d[key], (key, q[key], d[key])
        assert np.array_equal(sol.field(ea.FIELD_CELLTYPE), osim.field(orc.CELLTYPE))
        assert np.array_equal(sol.field(ea.FIELD_GRAINID), osim.field(orc.GRAINID))
