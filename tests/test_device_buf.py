"""The library's device buffers when memory runs out (tests/device_buf_check.hip,
compiled for the host with a runtime of its own)."""
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
    out = tmp_path_factory.mktemp("device_buf") / "device_buf_check"
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O1", "-std=c++17", "-Wall",
                    "-Wno-unused-function", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{REPO / 'include'}",
                    str(REPO / "tests" / "device_buf_check.hip"),
                    str(REPO / "cusr_amd" / "csrc" / "program.cpp"), "-pthread",
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    return out


@pytest.mark.parametrize("what", ["error", "room", "bound"])
def test_device_buffers(exe, what):
    r = subprocess.run([str(exe), what], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "device buffers ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
