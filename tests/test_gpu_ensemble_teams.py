"""GPU: an ensemble whose workgroups outnumber the compute units (hundreds of small domains, and larger
ones that get teams of several workgroups), stepped by launches of odd and large step counts; each
result compared with the same deck and seed run alone on the plain path."""
import numpy as np
import pytest

import exaca_amd as ea
from conftest import c_deck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks,steps", [(8, 50), (64, 1130)])
def test_more_workgroups_than_compute_units(tmp_path, blocks, steps):
    small = [c_deck(tmp_path / f"s{k}.txt", 6 + k % 5, nx=5 + k % 7, ny=4 + k % 3, density=5000, fraction=0.2)
             for k in range(35)]
    large = [c_deck(tmp_path / "l0.txt", 5, nx=90, ny=90, density=500), c_deck(tmp_path / "l1.txt", 4, nx=150, ny=120),
             c_deck(tmp_path / "l2.txt", 40, nx=40, ny=40, density=400)]
    jobs = [(small[k % 35], k + 1) for k in range(290)] + [(d, 7) for d in large]
    preps = [ea.Prepared(d, seed=s) for d, s in jobs]
    print(f"[ensemble teams] {len(jobs)} domains, at most {blocks} workgroups each, {steps} steps a call", flush=True)
    with ea.Ensemble(slots=len(jobs), arena_bytes=sum(p.device_bytes for p in preps) + (len(jobs) << 12)) as ens:
        ens.set_blocks(blocks)
        slots = [ens.admit(p) for p in preps]
        assert None not in slots
        for _ in range(400):
            ens.advance(steps)
            final, err = ens.poll_errors()
            assert not err.any(), err
            if (final > 0).all():
                break
        assert (final > 0).all()
        for k in list(range(0, 290, 29)) + [290, 291, 292]:
            q, slot = ens.query(slots[k]), slots[k]
            with ea.Solver(jobs[k][0], seed=jobs[k][1]) as sol:
                cycle, _ = sol.run()
                alone = sol.query()
                assert q["final_cycle"] == cycle, k
                assert [q[n] for n in ("nn", "frontier", "captures", "solidified")] == \
                       [alone[n] for n in ("nn", "frontier", "captures", "solidified")], k
                for field in (ea.FIELD_CELLTYPE, ea.FIELD_GRAINID):
                    assert np.array_equal(ens.field(slot, field, preps[k].cells), sol.field(field)), (k, field)
