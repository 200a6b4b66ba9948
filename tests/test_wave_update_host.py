"""The update and the wave speed in the wavefront forms (geoswe_amd/csrc/gs_wave.h) against the
general functions (gs_device.h), both built for the CPU (tests/native/wave_update_check.cpp):
wherever a form does not hand its row over, the values are equal, a NaN momentum in a cell that
has just become wet among them; the states of a flood are not handed over."""
import shutil
import subprocess
from pathlib import Path

import pytest

NATIVE = Path(__file__).resolve().parent / "native"


def test_update_forms_equal_general(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not available")
    exe = tmp_path / "wave_update_check"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-x", "hip", "-O2", "-std=c++17", "-ffp-contract=off", "-o",
                    str(exe), str(NATIVE / "wave_update_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "mismatches 0" in r.stdout
