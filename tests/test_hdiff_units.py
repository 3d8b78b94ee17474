"""What the LDS-DMA hdiff tile reads, checked on the host:
`hdiff_units_check.cpp` compiles against the tile's own header
(stencil_benchmarks_amd/csrc/hdiff_tile.h) and walks the units that it stages
over halos, extents and strides; none may leave the field."""

import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_hdiff_units_stay_in_the_field(tmp_path):
    exe = tmp_path / "hdiff_units_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-x", "hip", "--offload-arch=gfx950",
                    str(HERE / "hdiff_units_check.cpp"), "-o", str(exe)], check=True,
                   capture_output=True, timeout=300)
    done = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout + done.stderr
    assert done.stdout.startswith("ok:"), done.stdout
