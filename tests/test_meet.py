"""How a team's workgroups agree at the start of a launch (exaca_amd/csrc/meet.hpp), with a thread per
workgroup (tests/meet_check.cpp): whatever waits expire and however late some start, either all of them
take the domain or workgroup 0 alone does, so that no workgroup waits for one that does not run."""
import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(),
                    reason="hipcc not installed")
def test_a_team_meets_or_leaves_the_domain_to_one(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = tmp_path / "meet_check"
    subprocess.run([hipcc, "-O2", "-std=c++17", "--offload-arch=gfx950", "-I", str(REPO / "exaca_amd" / "csrc"),
                    str(REPO / "tests" / "meet_check.cpp"), "-o", str(exe), "-lpthread"], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
