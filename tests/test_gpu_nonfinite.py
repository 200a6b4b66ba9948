"""A NaN y-momentum in a dry cell that rain makes wet ends the step that meets it, with friction on
and off, in every sweep."""
import numpy as np
import pytest

from geoswe_amd import CompressedSolver, Config, Mesh2D, Solver2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout,dtype,compute", [
    (layout, dtype, None) for layout in ("dense", "dense-max", "flat", "flat-max", "chunks") for dtype in ("float32", "float64")
] + [("dense", "float32", "float64"), ("dense-max", "float32", "float64")])
@pytest.mark.parametrize("friction", ["none", "manning"])
def test_nan_momentum_in_a_cell_made_wet(gpu, friction, layout, dtype, compute):
    nx, ny = 9, 70
    q = np.zeros((3, nx, ny), dtype)
    q[0, :, :20] = 0.5
    cfg = Config(bc_x="fall", bc_y="fall", dtype=dtype, compute_dtype=compute, friction=friction,
                 manning_n=0.03 if friction == "manning" else 0.0, rainfall=1.0e-3)
    mesh = Mesh2D(nx, ny, 2.0, 2.0)
    s = Solver2D(mesh, cfg, q, np.zeros((nx, ny), dtype), track_max_depth=layout == "dense-max")
    at = (4, 40)
    if not layout.startswith("dense"):
        s = CompressedSolver.from_dense(s, cfl_linf=True, track_max_depth=layout == "flat-max")
        if layout == "chunks":
            s.traversal = "chunks"
        at = int(np.flatnonzero((s.fm.ij == np.array(at) + mesh.ngh).all(1))[0])
    plane = s._bufs[0][2].download()
    plane[at] = np.nan                            # the cell is dry: its momenta are not looked at yet
    s._bufs[0][2].upload(plane)
    with pytest.raises(FloatingPointError):
        s.advance(1)
