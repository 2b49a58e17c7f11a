"""An orientation file that is a pipe (a link to /dev/stdin among the substrates) is read like a regular one."""
import subprocess

from conftest import DATA, REPO


def test_orientations_from_a_pipe(tmp_path):
    csrc = REPO / "exaca_amd" / "csrc"
    exe = tmp_path / "orientations_pipe_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(csrc),
                    str(REPO / "tests" / "orientations_pipe_check.cpp"), str(csrc / "init.cpp"), str(csrc / "deck.cpp"),
                    "-o", str(exe), "-lpthread", "-ldl"], check=True, capture_output=True)
    path = DATA / "Substrate" / "GrainOrientationVectors_Robert.csv"
    r = subprocess.run([str(exe), str(path)], input=path.read_bytes(), capture_output=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
