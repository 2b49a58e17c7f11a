"""The growth over any run of steps by prefix sums per binade equals the step-by-step recurrence, bit
for bit (exaca_amd/csrc/growth.hpp; the cases are in tests/growth_steps_check.cpp)."""
import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(),
                    reason="hipcc not installed")
def test_growth_by_sums_matches_stepwise(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = tmp_path / "growth_steps_check"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950",
                    "-I", str(REPO / "exaca_amd" / "csrc"), str(REPO / "tests" / "growth_steps_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "mismatches 0" in r.stdout
