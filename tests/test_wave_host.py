"""The wavefront forms of the step arithmetic (geoswe_amd/csrc/gs_wave.h) against the general
functions (gs_device.h), both built for the CPU: tests/native/wave_check.cpp runs faces and
updates over wet states, films and dry cells on rough beds, flow beyond the friction velocity
cap, still water, and zeros, subnormals, huge values, infinities and NaN, in float32 and
float64. Wherever the wavefront form does not hand the row over, the values are equal; the
states of a flood are not handed over."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
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


@pytest.mark.parametrize("target", [1, 3, 7, 500, 4608])
def test_tile_height_rule_native_equals_python(monkeypatch, target):
    """The native mesh builder and the Python one pick the same tile height, where the square root
    decides (4000 to 12000 window rows) and at both clamps."""
    import geoswe_amd.flatmesh as FM
    monkeypatch.setattr(FM, "TILE_TARGET", target)
    for nx, ny in ((3, 61), (40, 121), (700, 400), (1000, 720)):
        inside = np.zeros((nx + 8, ny + 8), bool)
        inside[4:-4, 4:-4] = True
        a = FM.build_flat_mesh(inside, 4, native=True)
        b = FM.build_flat_mesh(inside, 4, native=False)
        assert np.array_equal(a.tile_irc, b.tile_irc) and np.array_equal(a.tile_e0, b.tile_e0)
        rows = FM.sweep_rows_for(nx * ((ny + 1) // 60 + 1))   # windows of the column grid that the rows touch
        tall = int(a.tile_irc[:, 1].max())
        assert tall == rows if nx > 2 * rows else tall <= rows    # bands are trimmed to the active rows
