"""GPU: the ensemble's autotuner tries each setting that differs once."""
import pytest

import exaca_amd as ea
from conftest import c_deck

pytestmark = pytest.mark.gpu


def test_autotuner_tries_each_setting_once(tmp_path):
    """A team has at most 64 workgroups: the settings tried are 16, 32 and 64, a chunk of 50 steps each."""
    prep = ea.Prepared(c_deck(tmp_path / "d.txt", 20, nx=60, ny=60, density=100))
    with ea.Ensemble(1, prep.device_bytes + (1 << 16)) as ens:
        slot = ens.admit(prep)
        assert ens.autotune(1) in (16, 32, 64)
        assert ens.query(slot)["steps"] == 3 * 50
        ens.set_blocks(256)  # accepted as before
        ens.advance(50)
        assert not ens.poll_errors()[1].any() and ens.query(slot)["steps"] == 200
