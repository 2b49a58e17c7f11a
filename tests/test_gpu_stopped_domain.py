"""GPU: a domain that an error stops. A team's barrier is given no time to wait, so that it gives up within the
first steps (every workgroup then leaves the kernel; nothing is touched by a workgroup that left): the
error is reported by the next check or poll, and no later call steps the domain any more."""
import numpy as np
import pytest

import exaca_amd as ea
from conftest import c_deck

pytestmark = pytest.mark.gpu


def test_a_barrier_that_gave_up_stops_the_domain(tmp_path, monkeypatch):
    deck = c_deck(tmp_path / "d.txt", 12, nx=56, ny=56, density=1000, fraction=0.3)
    monkeypatch.setenv("EXACA_BARRIER_US", "0")
    with ea.Solver(deck) as sol:
        assert sol.team()["workgroups"] == 8
        with pytest.raises(ea.ExacaError, match="16: a barrier wait"):
            sol.run(max_cycles=200)
        before = [sol.field(f) for f in (ea.FIELD_CELLTYPE, ea.FIELD_GRAINID)]
        assert (before[0] == 5).any()  # liquid left: a domain that were still stepped would change
        with pytest.raises(ea.ExacaError, match="16: a barrier wait"):
            sol.run(max_cycles=700)
        sol.step(701)
        with pytest.raises(ea.ExacaError, match="16: a barrier wait"):
            sol.check(701)
        for a, f in zip(before, (ea.FIELD_CELLTYPE, ea.FIELD_GRAINID)):
            assert np.array_equal(a, sol.field(f))


def test_an_ensemble_reports_a_barrier_that_gave_up(tmp_path, monkeypatch):
    monkeypatch.setenv("EXACA_BARRIER_US", "0")
    small = ea.Prepared(c_deck(tmp_path / "s.txt", 10, density=1000))
    large = ea.Prepared(c_deck(tmp_path / "l.txt", 12, nx=90, ny=90, density=1000, fraction=0.3))
    with ea.Ensemble(2, small.device_bytes + large.device_bytes + (1 << 16)) as ens:
        s, big = ens.admit(small), ens.admit(large)
        ens.advance(50)
        final, err = ens.poll_errors()
        assert err[big] == 16 and 1 <= final[big] <= 50 and ens.query(big)["error"] == 16
        ct = ens.field(big, ea.FIELD_CELLTYPE, large.cells)
        assert (ct == 5).any()
        ens.advance(500)
        again, err = ens.poll_errors()
        assert again[big] == final[big] and err[big] == 16 and ens.query(big)["final_cycle"] == final[big]
        assert np.array_equal(ct, ens.field(big, ea.FIELD_CELLTYPE, large.cells))
        # a team of one passes no barrier, whatever its bound
        assert err[s] in (0, 16)
