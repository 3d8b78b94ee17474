"""Launch rules of the register-column vadv, checked on the host:
`vadv_shape_check.cpp` compiles against the solver's own header
(stencil_benchmarks_amd/csrc/vadv_regs.h)."""

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_vadv_launch_rules(tmp_path):
    exe = tmp_path / "vadv_shape_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-x", "hip", "--offload-arch=gfx950",
                    str(HERE / "vadv_shape_check.cpp"), "-o", str(exe)], check=True,
                   capture_output=True, timeout=300)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout + done.stderr
    assert done.stdout.startswith("ok"), done.stdout
