"""The ensemble run that allocates nothing takes as many members as its header promises, 409 in
float32 and 384 in float64, and each steps as by itself; one more is refused."""
import numpy as np
import pytest

from geoswe_amd import CompressedSolver, Config, Mesh2D, Solver2D
from geoswe_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,most", [("float32", 409), ("float64", 384)])
def test_every_promised_member(gpu, dtype, most):
    from geoswe_amd.ensemble import run_noalloc
    nx, ny = 5, 6
    mesh = Mesh2D(nx, ny, 2.0, 2.0)
    cfg = Config(bc_x="fall", bc_y="fall", dtype=dtype, friction="manning", manning_n=0.03)
    bed = np.zeros((nx, ny), dtype)

    def member(k):
        q = np.zeros((3, nx, ny), dtype)
        q[0] = 0.2 + 0.001 * k
        q[0, 2, 3] += 0.1
        return CompressedSolver.from_dense(Solver2D(mesh, cfg, q, bed), cfl_linf=True, track_max_depth=False)

    members = [member(k) for k in range(most)]
    with pytest.raises(L.GsError, match="exceed"):
        run_noalloc(members + members[:1], 1)
    assert all(m.nsteps == 0 for m in members)
    run_noalloc(members, 2)
    for k in (0, 1, most // 2, most - 2, most - 1):
        one = member(k)
        one.advance(2)
        assert members[k].nsteps == 2 and members[k].t == one.t
        assert np.array_equal(members[k].q_flat(), one.q_flat())
