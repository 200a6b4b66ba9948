"""Films that friction has all but stopped, on the GPU: the sweep in wavefront forms against the
chunk traversal, which takes the general functions, bit for bit."""
import numpy as np
import pytest

from geoswe_amd import CompressedSolver, Config, Mesh2D, Solver2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("quadratic", [True, False])
@pytest.mark.parametrize("vcap", [15.0, 1.0e-20])
def test_creeping_films(gpu, vcap, quadratic, dtype):
    """Velocities of 1e-25 to 1e-8 m/s in still films of 1 um to 1 m, steps of 30 and 100 s."""
    nx, ny = 12, 130
    rng = np.random.default_rng(7)
    h = 10.0 ** rng.uniform(-5.9, 0.0, (nx, ny))
    u = 10.0 ** rng.uniform(-25.0, -8.0, (2, nx, ny)) * rng.choice([-1.0, 0.0, 1.0], (2, nx, ny))
    q = np.stack([h, h * u[0], h * u[1]]).astype(dtype)
    out = []
    for trav in ("tiles", "chunks"):
        cfg = Config(bc_x="wall", bc_y="wall", dtype=dtype, friction="manning", manning_n=0.1,
                     friction_quadratic_alpha=quadratic, friction_velocity_cap_ms=vcap)
        # the bed mirrors the films, so that the surface is level up to rounding
        s = Solver2D(Mesh2D(nx, ny, 2000.0, 2000.0), cfg, q, (2.0 - h).astype(dtype))
        c = CompressedSolver.from_dense(s, cfl_linf=True, track_max_depth=False, sweep_rows=3)
        c.traversal = trav
        for dt in (30.0, 100.0):
            c.step(dt)
        out.append(c.q_flat())
    assert np.array_equal(out[0], out[1])
