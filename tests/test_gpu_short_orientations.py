"""GPU: an orientation file with fewer rows than the domain has grains. The grains past its end have zero unit
vectors and critical lengths that are not numbers, which no half-diagonal reaches (the reference
compares with >=): they never capture, and the other grains grow around them. Every field and counter against
the oracle, by a team of one workgroup, of eight, and by two launches a step; and in an ensemble."""
import shutil

import numpy as np
import pytest

import exaca_amd as ea
import oracle as orc
from conftest import DATA, c_deck

pytestmark = pytest.mark.gpu


def _short_data(where, rows):
    shutil.copytree(DATA, where)
    f = where / "Substrate" / "GrainOrientationVectors_Robert.csv"
    f.write_text("\n".join(f.read_text().splitlines()[:1 + rows]) + "\n")
    return where


@pytest.mark.parametrize("side,rows,blocks", [(20, 3, None), (20, 0, None), (48, 40, None), (48, 40, 8)])
def test_grains_without_an_orientation_never_capture(tmp_path, monkeypatch, side, rows, blocks):
    if blocks:
        monkeypatch.setenv("EXACA_BLOCKS", str(blocks))
    data = _short_data(tmp_path / "data", rows)
    deck = c_deck(tmp_path / "d.txt", 10, nx=side, ny=side, density=2000, fraction=0.08)
    osim = orc.OracleSim(deck, data)
    osim.run(max_cycles=1500)
    with ea.Solver(deck, data_dir=data) as sol:
        sol.run(max_cycles=1500)
        q, d = sol.query(), osim.dims()
        assert d["nuclei"] > rows or (osim.field(orc.GRAINID) > rows).any()
        for key in ("nn", "captures", "solidified", "frontier"):
            assert q[key] == d[key], (key, q[key], d[key])
        assert (d["captures"] > 0) == (rows > 0)
        ct = sol.field(ea.FIELD_CELLTYPE)
        assert np.array_equal(ct, osim.field(orc.CELLTYPE))
        assert np.array_equal(sol.field(ea.FIELD_GRAINID), osim.field(orc.GRAINID))
        act = np.flatnonzero(ct == 2)
        assert np.array_equal(sol.field(ea.FIELD_DIAGONAL)[act], osim.field(orc.DIAGLEN)[act])


def test_in_an_ensemble(tmp_path):
    data = _short_data(tmp_path / "data", 40)
    deck = c_deck(tmp_path / "d.txt", 10, nx=48, ny=48, density=2000, fraction=0.08)
    prep = ea.Prepared(deck, data_dir=data)
    with ea.Ensemble(1, prep.device_bytes + (1 << 16)) as ens, ea.Solver(deck, data_dir=data) as sol:
        slot = ens.admit(prep)
        ens.advance(1500)
        assert not ens.poll_errors()[1].any()
        sol.run(max_cycles=1500)
        for f in (ea.FIELD_CELLTYPE, ea.FIELD_GRAINID):
            assert np.array_equal(ens.field(slot, f, prep.cells), sol.field(f))
