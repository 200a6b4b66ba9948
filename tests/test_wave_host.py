"""The wavefront forms of the step arithmetic (geoswe_amd/csrc/gs_wave.h) against the general
functions (gs_device.h), both built for the CPU: tests/native/wave_check.cpp runs faces and
updates over wet states, films and dry cells on rough beds, flow beyond the friction velocity
cap, still water, and zeros, subnormals, huge values, infinities and NaN, in float32 and
float64. Wherever the wavefront form does not hand the row over, the values are equal; the
states of a flood are not handed over."""
import shutil
import subprocess
from pathlib import Path

import pytest

NATIVE = Path(__file__).resolve().parent / "native"


def test_wave_forms_equal_general(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not available")
    exe = tmp_path / "wave_check"
    subprocess.run([hipcc, "--offload-arch=gfx950", "-x", "hip", "-O2", "-std=c++17", "-ffp-contract=off", "-o",
                    str(exe), str(NATIVE / "wave_check.cpp")], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "mismatches 0" in r.stdout
