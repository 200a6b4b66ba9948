"""The forcing tables of a step's plan, searched on the device, against the host's expressions."""
import bisect
import ctypes as C

import numpy as np
import pytest

from geoswe_amd import Config, Mesh2D, Solver2D, StageBoundary

pytestmark = pytest.mark.gpu


def _table(n, kind):
    rng = np.random.default_rng(n)
    t = np.cumsum(rng.random(n) + 0.05)
    if kind == "ties" and n > 3:
        t[n // 2] = t[n // 2 - 1]
        t[-1] = t[-2]
    return t, rng.random(n)


@pytest.mark.parametrize("kind", ["plain", "ties"])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 10, 17, 72, 81, 82, 401, 1000])
def test_rain_and_stage_of_a_plan_equal_the_host(gpu, n, kind):
    """Around, at and beyond table entries, with steps that stay in a segment and steps that pass
    over several, the planned rain segment and stage are bisect's and the host interpolation's."""
    from geoswe_amd import _lib as L
    ts, sv = _table(n, kind)
    keep = [L.DeviceArray.from_host(a) for a in (ts, sv, sv + 1.0, np.full(n, np.inf))]
    f = L.GsForcing()
    f.n_rain = f.n_stage = n
    f.rain_t = f.stage_t = keep[0].ptr
    f.stage_v, f.rain_rate, f.rain_cap = keep[1].ptr, keep[2].ptr, keep[3].ptr
    s = Solver2D(Mesh2D(4, 4, 1.0, 1.0), Config(bc_x="fall", bc_y="fall", dtype="float64"),
                 np.ones((3, 4, 4)), np.zeros((4, 4)))
    clk = s._clock
    sb = StageBoundary.__new__(StageBoundary)
    sb.time_s, sb.stage_m, sb._oor_warned = ts, sv, True
    rng = np.random.default_rng(n + 7)
    for t in np.concatenate([[0.0, ts[0], ts[-1], ts[-1] + 1.0], rng.choice(ts, 6), rng.random(8) * ts[-1],
                             np.nextafter(rng.choice(ts, 4), 0.0)]):
        for dt in (1e-9, 0.3, 1.7, 6.0, float(ts[-1])):
            L.call("gs_clock_reset", C.c_void_p(clk.ptr), C.c_double(float(t)), None)
            L.call("gs_clock_set_dt", C.c_void_p(clk.ptr), C.c_double(dt), C.byref(s._phys()), f, None)
            c = L.read_clock(clk)
            seg = min(max(bisect.bisect_right(ts.tolist(), float(t)) - 1, 0), n - 1)
            assert c.rain_idx == seg and c.rain32 == np.float32(sv[seg] + 1.0)
            assert c.eta64 == sb.stage_at_time(float(t) + dt), (t, dt)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("trav", ["tiles", "chunks"])
def test_frozen_steps_plan_the_next_dt(gpu, dtype, trav):
    """Steps whose plan takes the next frozen dt end in the state and the clock, byte for byte, of
    steps that are each given theirs; a dt of 0 among them (which a plan does not take) too."""
    from geoswe_amd import CompressedSolver, RainfallForcing, _lib as L
    rng = np.random.default_rng(11)
    nx, ny = 24, 70
    bed = rng.random((nx, ny))
    q = np.stack([np.maximum(1.0 - bed, 0), np.zeros((nx, ny)), np.zeros((nx, ny))])
    dts = np.array([0.01, 0.02, 0.015, 0.0, 0.03, 0.01])
    out = []
    for frozen in (True, False):
        mesh = Mesh2D(nx, ny, 2.0, 2.0)
        sea = np.zeros((nx, ny), bool)
        sea[0] = True
        sb = StageBoundary.from_mask(sea, mesh, bed, np.array([0.0, 0.02, 0.05, 1.0]), np.array([1.0, 1.3, 0.9, 1.1]))
        cfg = Config(bc_x="fall", bc_y="fall", dtype=dtype, friction="manning", manning_n=0.03, stage_boundary=sb,
                     rainfall_forcing=RainfallForcing(np.array([0.0, 0.03, 0.06]), np.array([10.0, 50.0, 0.0])))
        c = CompressedSolver.from_dense(Solver2D(mesh, cfg, q.astype(dtype), bed.astype(dtype)), cfl_linf=True,
                                        track_max_depth=False)
        c.traversal = trav
        if frozen:
            c._ensure_lam()
            L.call("gs_flat_run_frozen", C.byref(c._desc()), C.byref(c._phys()), c._fo.s, C.c_void_p(c._clock.ptr),
                   len(dts), C.c_void_p(dts.ctypes.data), None, 0, None, 1, None, None)
            L.sync(None)
        else:
            c._ensure_lam()
            for dt in dts:
                L.call("gs_clock_set_dt", C.c_void_p(c._clock.ptr), C.c_double(dt), C.byref(c._phys()), c._fo.s, None)
                L.call("gs_flat_step", C.byref(c._desc()), C.byref(c._phys()), c._fo.s, C.c_void_p(c._clock.ptr), None)
            L.sync(None)
        out.append((c.q_flat(), c._clock.download().tobytes(), c.nsteps))
    assert out[0][2] == out[1][2] == len(dts)
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]


@pytest.mark.parametrize("trav,ga", [("tiles", False), ("chunks", False), ("tiles", True)])
@pytest.mark.parametrize("n", [1, 2, 5])
def test_frozen_steps_sample_the_gauges(gpu, trav, ga, n):
    """The depths after every frozen step at 1, 64 and 130 gauges (repeated ids among them), whether
    the next step's sweep samples them or a launch does, are the depths of steps taken one by one."""
    from geoswe_amd import CompressedSolver, _lib as L
    rng = np.random.default_rng(3)
    nx, ny = 20, 66
    bed = rng.random((nx, ny))
    q = np.stack([np.maximum(1.2 - bed, 0), np.zeros((nx, ny)), np.zeros((nx, ny))]).astype(np.float32)
    dts = np.full(n, 0.01)

    def solver():
        cfg = Config(bc_x="fall", bc_y="fall", dtype="float32", friction="manning", manning_n=0.03)
        c = CompressedSolver.from_dense(Solver2D(Mesh2D(nx, ny, 2.0, 2.0), cfg, q, bed.astype(np.float32)),
                                        cfl_linf=True, track_max_depth=ga)     # the maximum: not the lean sweep
        c.traversal = trav
        c._ensure_lam()
        return c

    ref = solver()
    want = []
    for dt in dts:
        ref.step(dt)
        want.append(ref.q_flat()[0])
    for g in (1, 64, 130):
        c = solver()
        ids = rng.choice(np.flatnonzero(c.fm.active), size=g)
        d_ids, out = L.DeviceArray.from_host(ids.astype(np.int64)), L.DeviceArray((n, g), np.float32, zero=True)
        L.call("gs_flat_run_frozen", C.byref(c._desc()), C.byref(c._phys()), c._fo.s, C.c_void_p(c._clock.ptr), n,
               C.c_void_p(dts.ctypes.data), C.c_void_p(d_ids.ptr), g, C.c_void_p(out.ptr), 1, None, None)
        L.sync(None)
        assert np.array_equal(out.download(), np.stack([w[ids] for w in want]))
