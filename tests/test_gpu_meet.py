"""GPU: launches of a team whose workgroups do not all run at once. With no time to meet, every launch is left
to one workgroup of the team; with 1 us, some are: a domain stepped so equals the oracle, and an ensemble
equals one whose teams meet. Two ensembles that each fill the compute units and a solver, stepped
from three threads at once, all end, with the results they have alone."""
import threading

import numpy as np
import pytest

import exaca_amd as ea
import oracle as orc
from conftest import DATA, c_deck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wait", [0, 1])
@pytest.mark.parametrize("side,workgroups", [(44, 8), (70, 16), (96, 32)])
def test_domain_left_to_one_workgroup_matches_the_oracle(tmp_path, monkeypatch, side, workgroups, wait):
    monkeypatch.setenv("EXACA_MEET_US", str(wait))
    deck = c_deck(tmp_path / "d.txt", 8, nx=side, ny=side, density=1000, fraction=0.2)
    osim = orc.OracleSim(deck, DATA)
    osim.run(max_cycles=300)
    with ea.Solver(deck) as sol:
        for c in (1, 2, 3, 40, 41, 173, 174, 175, 300):
            sol.run(max_cycles=c)
        team = sol.team()
        print(f"[meet] {side}: {team}", flush=True)
        assert team["workgroups"] == workgroups and team["launches"] == 9
        assert team["alone"] == 9 if wait == 0 else 0 <= team["alone"] <= 9
        q, d = sol.query(), osim.dims()
        for key in ("nn", "captures", "solidified", "frontier"):
            assert q[key] == d[key], (key, q[key], d[key])
        ct = sol.field(ea.FIELD_CELLTYPE)
        assert np.array_equal(ct, osim.field(orc.CELLTYPE))
        assert np.array_equal(sol.field(ea.FIELD_GRAINID), osim.field(orc.GRAINID))
        act = np.flatnonzero(ct == 2)
        assert np.array_equal(sol.field(ea.FIELD_DIAGONAL)[act], osim.field(orc.DIAGLEN)[act])


def test_bad_waits_are_refused(tmp_path, monkeypatch):
    deck = c_deck(tmp_path / "d.txt", 8)
    for bad in ("-1", "x", "", "40000001"):
        monkeypatch.setenv("EXACA_MEET_US", bad)
        with pytest.raises(ea.ExacaError, match="EXACA_MEET_US"):
            ea.Solver(deck)
        with pytest.raises(ea.ExacaError, match="EXACA_MEET_US"):
            ea.Ensemble(1, 1 << 20)


def _solve_all(preps, steps):
    with ea.Ensemble(len(preps), sum(p.device_bytes for p in preps) + (len(preps) << 12)) as ens:
        slots = [ens.admit(p) for p in preps]
        for _ in range(200):
            ens.advance(steps)
            final, err = ens.poll_errors()
            assert not err.any(), err
            if (final > 0).all():
                break
        assert (final > 0).all()
        out = []
        for s, p in zip(slots, preps):
            q = ens.query(s)
            out.append((int(final[s]), [q[n] for n in ("nn", "frontier", "captures", "solidified")],
                        ens.field(s, ea.FIELD_CELLTYPE, p.cells), ens.field(s, ea.FIELD_GRAINID, p.cells)))
        return out


def _same(a, b):
    for k, (x, y) in enumerate(zip(a, b)):
        assert x[:2] == y[:2], k
        assert np.array_equal(x[2], y[2]) and np.array_equal(x[3], y[3]), k


def _domains(tmp_path, tag, count, seed):
    decks = [c_deck(tmp_path / f"{tag}{k}.txt", 6 + k % 9, nx=24 + 9 * (k % 8), ny=70 - 7 * (k % 7), density=800,
                    fraction=0.1) for k in range(count)]
    return [ea.Prepared(d, seed=seed + k) for k, d in enumerate(decks)]


def test_ensemble_left_to_single_workgroups(tmp_path, monkeypatch):
    preps = _domains(tmp_path, "e", 24, 5)
    met = _solve_all(preps, 400)
    for wait in ("0", "1", "3"):
        monkeypatch.setenv("EXACA_MEET_US", wait)
        print(f"[meet] ensemble with {wait} us to meet", flush=True)
        _same(_solve_all(preps, 400), met)


def test_ensembles_and_a_solver_at_once(tmp_path):
    a, b = _domains(tmp_path, "a", 40, 100), _domains(tmp_path, "b", 48, 900)
    deck = c_deck(tmp_path / "s.txt", 60, nx=96, ny=90, density=100)
    alone = [_solve_all(a, 150), _solve_all(b, 100)]

    def solver():
        with ea.Solver(deck) as sol:
            cycle, _ = sol.run()
            return cycle, sol.field(ea.FIELD_CELLTYPE), sol.field(ea.FIELD_GRAINID)

    single = solver()
    print("[meet] two ensembles and a solver at once", flush=True)
    got, failed = {}, []

    def go(name, f):
        try:
            got[name] = f()
        except BaseException as e:  # noqa: B902 -- reported by the test's own thread
            failed.append((name, e))

    threads = [threading.Thread(target=go, args=x) for x in
               (("a", lambda: _solve_all(a, 150)), ("b", lambda: _solve_all(b, 100)), ("s", solver))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    _same(got["a"], alone[0])
    _same(got["b"], alone[1])
    assert got["s"][0] == single[0] and all(np.array_equal(x, y) for x, y in zip(got["s"][1:], single[1:]))
