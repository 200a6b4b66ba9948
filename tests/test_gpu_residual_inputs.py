"""The dense residual takes the fluxes and the inactive cells alone: rain, the Manning number, its
classes and its field leave it as it is, in both precisions and at both offset widths of the sweep
(a tile height of 1 << 25 rows takes 64-bit offsets)."""
import numpy as np
import pytest

from geoswe_amd import Config, Mesh2D, RainfallForcing, Solver2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("rows", [3, 1 << 25])
@pytest.mark.parametrize("masked", [False, True])
def test_residual_without_rain_and_friction(gpu, masked, rows, dtype):
    nx, ny = 11, 125
    rng = np.random.default_rng(5)
    bed = rng.random((nx, ny)).astype(dtype)
    q = np.stack([np.maximum(0.8 - bed, 0.0), 0.1 * rng.random((nx, ny)), 0.1 * rng.random((nx, ny))]).astype(dtype)
    mesh = Mesh2D(nx, ny, 2.0, 2.0)
    cls = rng.integers(0, 40, (nx, ny)).astype(np.uint8)

    def residual(rain, manning):
        kw = {"gridded": dict(rainfall_forcing=RainfallForcing(np.array([0.0]), 1.0e4 * rng.random((1, nx, ny)))),
              "uniform": dict(rainfall=1.0e-3), None: {}}[rain]
        if manning:
            kw.update(friction="manning", manning_n=0.03)
        s = Solver2D(mesh, Config(bc_x="wall", bc_y="fall", dtype=dtype, **kw), q, bed, tile_rows=rows)
        if manning == "classes":
            s.set_manning_table(np.pad(cls, mesh.ngh, mode="edge"), np.linspace(0.02, 0.09, 40))
        elif manning == "field":
            s.set_manning(0.02 + 1e-3 * rng.random((nx, ny)))
        if masked:
            s.set_inside_mask(cls > 2)
        return s.residual()

    want = residual(None, None)
    assert np.abs(want).max() > 0.0
    for rain in ("uniform", "gridded"):
        for manning in ("number", "classes", "field"):
            assert np.array_equal(residual(rain, manning), want), (rain, manning)
