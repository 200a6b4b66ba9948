"""The launch query names the grid of the step: one wavefront per tile and, where the sweep forces the
ring cells itself, the workgroups that do (a multiple of 8)."""
import numpy as np
import pytest

from geoswe_amd import CompressedSolver, Config, Mesh2D, Solver2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,waves", [("float32", 8), ("float64", 4)])
@pytest.mark.parametrize("kind", ["lean", "sponge", "sponge-ext"])
def test_grid_of_tiles_and_ring_cells(gpu, kind, dtype, waves):
    nx, ny = 300, 700
    mesh = Mesh2D(nx, ny, 2.0, 2.0)
    q = np.zeros((3, nx, ny), dtype)
    q[0] = 0.5
    s = Solver2D(mesh, Config(bc_x="fall", bc_y="fall", dtype=dtype), q, np.zeros((nx, ny), dtype))
    c = CompressedSolver.from_dense(s, cfl_linf=True, track_max_depth=False, sweep_rows=5)
    shape = (c.fm.nxp, c.fm.nyp)
    if kind != "lean":
        c.set_sponge({"keep": np.full(shape, 0.9), "amb": np.zeros(shape)})
    if kind == "sponge-ext":
        c.set_ga_drain({"cls_pad": np.zeros(shape, np.uint8), "Ks_t": [1e-5], "psi_t": [0.1], "dth_t": [0.3],
                        "F_pad": None, "inv_tau_pad": None, "mode": "fused"})
    ring = 0 if kind == "lean" else c.n_stored - c.n_active
    per = -(-ring // (64 * waves))
    info = c.launch_info()
    assert info["kernel"] == ("sweep_ext" if kind == "sponge-ext" else "sweep")
    assert info["blocks"] == -(-len(c.fm.tile_e0) // waves) + -(-per // 8) * 8
