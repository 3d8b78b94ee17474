"""The staged device-to-host copy, checked on the host: `staged_copy_check.cpp`
compiles against the library's own source
(stencil_benchmarks_amd/csrc/runtime.hip) with host functions in place of the
HIP calls."""

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_staged_copy(tmp_path):
    exe = tmp_path / "staged_copy_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-x", "hip", "--offload-arch=gfx950",
                    "-Wno-everything", str(HERE / "staged_copy_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=300)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout + done.stderr
    assert done.stdout.startswith("ok"), done.stdout
