"""What the host plans a launch's LDS and indices by, against what the device uses
(tests/layout_check.hip, compiled for the host)."""
import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("layout") / "layout_check"
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-Wall",
                    "-Wno-unused-function", "-ffp-contract=off", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", f"-I{REPO / 'include'}",
                    str(REPO / "tests" / "layout_check.hip"),
                    str(REPO / "cusr_amd" / "csrc" / "program.cpp"), "-pthread", "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    return out


@pytest.mark.parametrize("what", ["eval", "solve", "scalars", "limit", "long", "order", "kept"])
def test_layout(exe, what):
    r = subprocess.run([str(exe), what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "layout ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
