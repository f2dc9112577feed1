"""The staged programs the device runs against the plain ones of co_decode, on
the host: same bits for values, tangents and adjoints, and every index within
the rows, slots and tapes that size the device's LDS (tests/staged_check.cpp)."""
import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]


def test_staged_programs_match_plain(tmp_path):
    exe = tmp_path / "staged_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wno-unused-function", "-pthread",
                    "-ffp-contract=off", "-D__host__=", "-D__device__=", "-o", str(exe),
                    str(REPO / "tests" / "staged_check.cpp"),
                    str(REPO / "cusr_amd" / "csrc" / "program.cpp")], check=True)
    r = subprocess.run([str(exe), "400"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "staged ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
