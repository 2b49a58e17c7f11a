"""GPU: a domain that an error stops. A team's barrier is given no time to wait, so that it gives up within the
first steps (every workgroup then leaves the kernel; nothing is touched by a workgroup that left): the
error is reported by the next check or poll, and no later call steps the domain any more."""
import numpy as np
import pytest

import exaca_amd as ea
from conftest import c_deck, s_deck

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


def _zero_grain_deck(where, radius):
    """A spot deck whose substrate file gives GrainID 0 to a quarter of the plane: the kernels flag its
    active cells (error 2) when they first look at their critical lengths."""
    deck = s_deck(where / "spot.txt", nsx=1, nsy=1, offset=2 * radius, radius=radius, density=50, spacing=8)
    side, nz = 4 + 2 * radius, radius + 3
    lines = [f"nz = {nz}", f"ny = {side}", f"nx = {side}"]
    for _ in range(nz):
        for j in range(side):
            lines += [str(0 if i < side // 2 and j < side // 2 else 1 + (7 * i + j) % 50) for i in range(side)]
    (where / "substrate.txt").write_text("\n".join(lines) + "\n")
    text = deck.read_text().splitlines()
    at = next(k for k, ln in enumerate(text) if ln.startswith("Substrate grain spacing"))
    text[at:at + 1] = [f"Path to substrate file: {where}", "Substrate file name: substrate.txt"]
    deck.write_text("\n".join(text) + "\n")
    return deck


@pytest.mark.parametrize("radius,workgroups", [(12, 1), (32, 8), (12, 0)])
def test_an_error_stops_the_domain_at_its_step(tmp_path, monkeypatch, radius, workgroups):
    """The state and the counters after many steps asked for at once are those at the end of the step that raised
    the flag (found by steps of one call each), and stay so."""
    if not workgroups:
        monkeypatch.setenv("EXACA_BLOCKS", "8")
    deck = _zero_grain_deck(tmp_path, radius)
    keys = ("nn", "frontier", "captures", "solidified", "waiting", "evaluated", "masks")

    def look(sol):
        q = sol.query()
        return [q[k] for k in keys], [sol.field(f) for f in (ea.FIELD_CELLTYPE, ea.FIELD_GRAINID, ea.FIELD_DIAGONAL)]

    with ea.Solver(deck) as sol:
        assert sol.team()["workgroups"] == workgroups
        for stop in range(1, 1000):
            sol.step(stop)
            try:
                sol.check(stop)
            except ea.ExacaError as e:
                assert "2: an active cell with GrainID 0" in str(e)
                break
        assert stop < 900
        want = look(sol)
    print(f"[stopped] radius {radius}, {workgroups} workgroups: step {stop}", flush=True)
    for end in (900, 901):
        with ea.Solver(deck) as sol:
            with pytest.raises(ea.ExacaError, match="2: an active cell with GrainID 0"):
                sol.run(max_cycles=end)
            for _ in range(2):
                got = look(sol)
                assert got[0] == want[0], (end, dict(zip(keys, got[0])), dict(zip(keys, want[0])))
                for a, b in zip(got[1], want[1]):
                    assert np.array_equal(a, b)
                sol.step(end + 1)  # the domain has ended: nothing changes any more
                end += 1
