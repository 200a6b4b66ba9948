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
