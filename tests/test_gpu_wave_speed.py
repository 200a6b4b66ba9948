"""Every wave speed of the flat sweeps: the L-inf norm, the L2 norm (the default of
CompressedSolver.from_dense), and both with a CFL floor above h_min. The sweep's rows take the
wavefront forms under each of them and give the chunk traversal's bits, states that the forms do
not take among them; ensemble members equal their plain runs."""
import numpy as np
import pytest

from geoswe_amd import CompressedSolver, Config, Mesh2D, Solver2D

pytestmark = pytest.mark.gpu

SPEEDS = [dict(cfl_linf=True), dict(), dict(cfl_linf=True, h_min_cfl=1.0e-3), dict(h_min_cfl=0.02)]


def _state(nx, ny, dtype, odd):
    rng = np.random.default_rng(nx * 1000 + ny)
    bed = (rng.random((nx, ny)) * 1.2).astype(dtype)
    h = np.maximum(0.8 - bed, 0.0).astype(dtype)
    q = np.stack([h, (rng.random((nx, ny)) - 0.5) * h, (rng.random((nx, ny)) - 0.5) * h]).astype(dtype)
    if odd:
        i, j = rng.integers(0, nx, 4), rng.integers(0, ny, 4)
        q[0, i, j] = 0.5
        q[1, i[0], j[0]] = 4.0e3
        q[2, i[1], j[1]] = -1.0e-42
        q[0, i[2], j[2]] = 1.0e-33
        bed[i[3], j[3]] = 3.0e6
    return q, bed, rng


def _solver(shape, rows, speed, dtype, odd, maxh, ext, h_min=None):
    nx, ny = shape
    q, bed, rng = _state(nx, ny, dtype, odd)
    cfg = Config(bc_x="fall", bc_y="fall", dtype=dtype, friction="manning", manning_n=0.03, rainfall=20.0 / 3.6e6,
                 **({} if h_min is None else {"h_min": h_min}))
    s = Solver2D(Mesh2D(nx, ny, 2.0, 2.0), cfg, q, bed)
    mask = rng.random((nx, ny)) > 0.06
    mask[nx // 2, ny // 2] = True
    s.set_inside_mask(mask)
    c = CompressedSolver.from_dense(s, track_max_depth=maxh, sweep_rows=rows, **speed)
    if ext:
        full = (nx + 2 * s.mesh.ngh, ny + 2 * s.mesh.ngh)
        c.set_ga_drain({"cls_pad": np.zeros(full, np.uint8), "Ks_t": [2e-5], "psi_t": [0.1], "dth_t": [0.3],
                        "F_pad": None, "inv_tau_pad": np.full(full, 1.0 / 600.0), "mode": "fused"})
    return c


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("maxh,ext", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("speed", SPEEDS)
@pytest.mark.parametrize("shape,rows", [((17, 61), 2), ((40, 130), 7), ((2100, 70), 1)])
def test_tiles_equal_chunks(gpu, shape, rows, speed, maxh, ext, dtype, odd):
    out = []
    for trav in ("tiles", "chunks"):
        c = _solver(shape, rows, speed, dtype, odd, maxh, ext)
        c.traversal = trav
        c.advance(3)
        out.append((c.q_flat(), c.t, c.nsteps, c._clockv().lam_bits, c.max_depth() if maxh else None))
    a, b = out
    assert a[1:4] == b[1:4] and np.array_equal(a[0], b[0])
    assert not maxh or np.array_equal(a[4], b[4])


@pytest.mark.parametrize("dtype,h_min", [("float32", 1.0e-7), ("float64", 1.0e-13)])
@pytest.mark.parametrize("maxh,ext", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("speed", SPEEDS[:2])
@pytest.mark.parametrize("shape,rows", [((17, 61), 2), ((2100, 70), 1)])
def test_dry_floors_that_the_forms_do_not_take(gpu, shape, rows, speed, maxh, ext, dtype, h_min):
    """Below 2^-21 (float32) and 2^-36 (float64) the sweeps step by the general functions alone."""
    out = []
    for trav in ("tiles", "chunks"):
        c = _solver(shape, rows, speed, dtype, False, maxh, ext, h_min)
        c.traversal = trav
        c.advance(3)
        out.append((c.q_flat(), c.t, c._clockv().lam_bits))
    assert out[0][1:] == out[1][1:] and np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("maxh", [False, True])
def test_ensemble_of_every_wave_speed(gpu, maxh, dtype):
    from geoswe_amd.ensemble import Ensemble
    for speeds in (SPEEDS, SPEEDS[1:2] * 3):
        members, plain = ([_solver((17 + 9 * k, 61 + 30 * k), 3, speed, dtype, False, maxh, False)
                           for k, speed in enumerate(speeds)] for _ in range(2))
        e = Ensemble(members, graph_batch=2)
        e.advance(5)
        for m, p in zip(members, plain):
            p.advance(5)
            assert m.t == p.t and np.array_equal(m.q_flat(), p.q_flat())
        e.close()


@pytest.mark.parametrize("speed", SPEEDS)
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("shape,rows", [((40, 130), 7), ((2100, 70), 1)])
def test_pre_friction_state(gpu, shape, rows, dtype, speed):
    """The adjoint's recomputing step of each wave speed makes the plain step's state."""
    import ctypes as C
    from geoswe_amd import _lib as L
    a, b = (_solver(shape, rows, speed, dtype, False, False, False) for _ in range(2))
    pre = [L.DeviceArray((a.n_stored,), a.dtype, zero=True) for _ in range(3)]
    for s in (a, b):
        p = C.byref(s._phys())
        L.call("gs_clock_reset", C.c_void_p(s._clock.ptr), C.c_double(0.0), None)
        L.call("gs_clock_set_dt", C.c_void_p(s._clock.ptr), C.c_double(0.01), p, s._fo.s, None)
        if s is a:
            L.call("gs_flat_step_pre", C.byref(s._desc()), p, s._fo.s, C.c_void_p(s._clock.ptr),
                   *[C.c_void_p(x.ptr) for x in pre], None)
        else:
            L.call("gs_flat_step", C.byref(s._desc()), p, s._fo.s, C.c_void_p(s._clock.ptr), None)
    L.sync(None)
    assert np.array_equal(a.q_flat(), b.q_flat()) and a._clockv().lam_bits == b._clockv().lam_bits
    assert (pre[0].download()[a.fm.active] > 0).any()


def test_float64_members_at_one_height(gpu):
    """Float64 members whose own tile heights differ (3, 1 and 2 rows) step at the height their total
    calls for, with their own tables left as they are; a height that the caller gave a member stays."""
    from geoswe_amd.ensemble import Ensemble
    from geoswe_amd.flatmesh import sweep_rows_for64
    shapes = ((110, 3700), (40, 130), (60, 1200), (30, 200))
    members, plain = ([_solver(sh, 5 if k == 3 else None, SPEEDS[0], "float64", False, False, False)
                       for k, sh in enumerate(shapes)] for _ in range(2))
    own = [int(m.fm.tile_irc[:, 1].max()) for m in members]
    assert own == [3, 1, 2, 5]
    rows = sweep_rows_for64(sum(int(m.fm.tile_irc[:, 1].sum()) for m in members))
    assert rows == 3
    e = Ensemble(members, graph_batch=2)
    assert e.sweep_rows == rows and len(e._tiles) == 2      # the second and the third member
    assert [int(m.fm.tile_irc[:, 1].max()) for m in members] == own
    e.advance(5)
    for m, p in zip(members, plain):
        p.advance(5)
        assert m.t == p.t and np.array_equal(m.q_flat(), p.q_flat())
    e.close()
