"""What the host plans a launch's LDS and indices by, against what the device uses
(tests/layout_check.cpp, on the host)."""
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("layout") / "layout_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wno-unused-function", "-pthread",
                    "-ffp-contract=off", "-D__host__=", "-D__device__=", "-o", str(out),
                    str(REPO / "tests" / "layout_check.cpp"),
                    str(REPO / "cusr_amd" / "csrc" / "program.cpp")], check=True)
    return out


@pytest.mark.parametrize("what", ["eval", "solve"])
def test_layout(exe, what):
    r = subprocess.run([str(exe), what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "layout ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
