"""The dense step with 64-bit offsets, which loads a cell's flags, class, Manning field, rain frame and
running maximum at their use, against the step that loads them a row ahead with 32-bit offsets:
the same bits. The 64-bit step is the one whose tiles reach 2 GiB, counted as if every tile were
full, so a tile height of 1 << 25 rows takes it on a grid of any width."""
import numpy as np
import pytest

from geoswe_amd import Config, Mesh2D, RainfallForcing, Solver2D, StageBoundary

pytestmark = pytest.mark.gpu

WIDE = 1 << 25


@pytest.mark.parametrize("dtype,compute", [("float32", None), ("float64", None), ("float32", "float64")])
@pytest.mark.parametrize("manning", ["number", "flags", "plane", "field"])
@pytest.mark.parametrize("gridded,masked,maxh", [(False, False, True), (True, False, False), (False, True, False),
                                                 (True, True, True)])
@pytest.mark.parametrize("shape,rows", [((5, 61), 1), ((23, 130), 4)])
def test_wide_step_equals_planes_loaded_ahead(gpu, shape, rows, gridded, masked, maxh, manning, dtype, compute):
    nx, ny = shape
    rng = np.random.default_rng(nx + ny)
    bed = (rng.random((nx, ny)) * 1.2).astype(dtype)
    h = np.maximum(0.8 - bed, 0.0).astype(dtype)
    q = np.stack([h, (rng.random((nx, ny)) - 0.5) * h, (rng.random((nx, ny)) - 0.5) * h]).astype(dtype)
    mask = rng.random((nx, ny)) > 0.1
    frames = rng.random((2, nx, ny)) * 4.0e4
    cls = rng.integers(0, 40 if manning == "plane" else 5, (nx, ny)).astype(np.uint8)
    n_of = np.linspace(0.02, 0.09, 40 if manning == "plane" else 5)
    mesh = Mesh2D(nx, ny, 2.0, 2.0, ngh=4)
    sea = np.zeros((nx, ny), bool)
    sea[:, 0] = True
    out = []
    for tile_rows in (rows, WIDE):
        kw = dict(rainfall_forcing=RainfallForcing(np.array([0.0, 2e-3]), frames)) if gridded else \
            dict(rainfall=20.0 / 3.6e6)
        if masked:
            kw["stage_boundary"] = StageBoundary.from_mask(sea, mesh, bed, np.array([0.0, 1.0]), np.array([0.9, 1.4]))
        cfg = Config(bc_x="fall", bc_y="wall", dtype=dtype, compute_dtype=compute, friction="manning",
                     manning_n=0.03, **kw)
        s = Solver2D(mesh, cfg, q, bed, tile_rows=tile_rows, track_max_depth=maxh)
        wide = s.pitch * np.dtype(dtype).itemsize >= (1 << 31) // tile_rows
        assert wide == (tile_rows == WIDE)
        if manning == "field":
            s.set_manning(n_of[cls] + 1e-3 * np.arange(ny))
        elif manning != "number":
            s.set_manning_table(np.pad(cls, 4, mode="edge"), n_of)
        if masked:
            s.set_inside_mask(mask)
            s.set_cfl_ghost_mask(~mask)
        for dt in (1e-3, 2e-3, 1e-3):
            s.step(dt)
        out.append((s.q_interior, s.max_depth() if maxh else None, s._clockv().lam_bits))
    a, b = out
    assert np.array_equal(a[0], b[0]) and a[2] == b[2]
    assert not maxh or np.array_equal(a[1], b[1])
