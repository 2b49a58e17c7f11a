"""The compiled barrier of a team of workgroups (k_steps, k_steps_n): its release is a write-back of the
L2, which is done only when the wave has waited for it. The device code is compiled as the library is and
read: between every write-back and the store of the barrier's word, and in every wave before the
workgroup's barrier that the write-back follows, stands a wait for all outstanding memory operations."""
import re
import subprocess

import pytest

from exaca_amd import build

MEMORY = re.compile(r"\s*(global|flat|buffer|scratch)_")
WAIT = re.compile(r"\s*s_waitcnt\b.*\bvmcnt\(0\)")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "k.s"
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "--cuda-device-only", "-S", str(build.CSRC / "ca_kernels.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    body, found = [], {}
    for line in out.read_text().splitlines():
        body.append(line)
        m = re.match(r"\s*\.end_amdhsa_kernel", line)
        if m:
            name = next(ln.split()[1] for ln in body if ".amdhsa_kernel" in ln)
            found[name] = body
            body = []
    teams = {n: b for n, b in found.items() if re.search(r"7k_steps|9k_steps_n", n)}
    assert len(teams) == 2
    return teams


def _first(lines, *patterns):
    """The first line that one of the patterns matches, and which."""
    for line in lines:
        for k, p in enumerate(patterns):
            if p.match(line):
                return k, line
    return None, None


def test_write_back_is_waited_for(kernels):
    for name, body in kernels.items():
        at = [i for i, line in enumerate(body) if "buffer_wbl2" in line]
        assert at, name
        for i in at:
            k, line = _first(body[i + 1:], WAIT, MEMORY)
            assert k == 0, f"{name}: {line.strip()} follows the write-back without a wait"


def test_every_wave_drains_before_the_release(kernels):
    barrier = re.compile(r"\s*s_barrier")
    for name, body in kernels.items():
        for i in (i for i, line in enumerate(body) if "buffer_wbl2" in line):
            back = body[i - 1::-1]
            k = next(k for k, line in enumerate(back) if barrier.match(line))
            w, line = _first(back[k + 1:], WAIT, MEMORY)
            assert w == 0, f"{name}: {line.strip()} may be outstanding at the barrier before the write-back"


def test_invalidation_is_waited_for(kernels):
    barrier = re.compile(r"\s*s_barrier")
    for name, body in kernels.items():
        at = [i for i, line in enumerate(body) if "buffer_inv" in line]
        assert at, name
        for i in at:
            k, line = _first(body[i + 1:], WAIT, MEMORY, barrier)
            assert k == 0, f"{name}: {line.strip()} follows the invalidation without a wait"
