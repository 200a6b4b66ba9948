"""Frozen-dt runs (gs_flat_run_frozen) against the same steps one by one: the depths at listed cells
"after every step" are those that gs_flat_sample reads after gs_flat_step, at cells of the ring too,
which the next step's ring mode overwrites in its input state."""
import ctypes as C

import numpy as np
import pytest

from geoswe_amd import CompressedSolver, Config, Mesh2D, Solver2D
from geoswe_amd import _lib as L

pytestmark = pytest.mark.gpu

DTS = np.array([0.02, 0.05, 0.03, 0.04, 0.01])


def _solver(dtype, mode, maxh):
    nx, ny = 20, 75
    rng = np.random.default_rng(3)
    bed = (0.4 * rng.random((nx, ny))).astype(dtype)
    q = np.stack([np.maximum(0.8 - bed, 0.0), 0.1 * rng.random((nx, ny)), 0.1 * rng.random((nx, ny))]).astype(dtype)
    cfg = Config(bc_x="fall", bc_y="fall", dtype=dtype, friction="manning", manning_n=0.03)
    s = Solver2D(Mesh2D(nx, ny, 2.0, 2.0), cfg, q, bed)
    mask = np.ones((nx, ny), bool)
    mask[:, 40:44] = False
    s.set_inside_mask(mask)
    c = CompressedSolver.from_dense(s, cfl_linf=True, track_max_depth=maxh)
    if mode:
        c.set_ring_mode(mode, eta=1.1)
    return c


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("maxh", [False, True])
@pytest.mark.parametrize("mode", [None, "stage", "extrapolate"])
def test_samples_are_the_depths_after_each_step(gpu, mode, maxh, dtype):
    a, b = _solver(dtype, mode, maxh), _solver(dtype, mode, maxh)
    ring = a._rmode["ids"].download()[::7] if mode else np.flatnonzero(~a.fm.active)[::9]
    ids = np.sort(np.concatenate([ring, np.flatnonzero(a.fm.active)[::50]])).astype(np.int64)
    d_ids = L.DeviceArray.from_host(ids)
    got = L.DeviceArray((len(DTS), len(ids)), a.dtype, zero=True)
    want = L.DeviceArray((len(DTS), len(ids)), a.dtype, zero=True)
    es = np.dtype(a.dtype).itemsize
    for s in (a, b):
        L.call("gs_clock_reset", C.c_void_p(s._clock.ptr), C.c_double(0.0), None)
    L.call("gs_flat_run_frozen", C.byref(a._desc()), C.byref(a._phys()), a._fo.s, C.c_void_p(a._clock.ptr), len(DTS),
           C.c_void_p(DTS.ctypes.data), C.c_void_p(d_ids.ptr), len(ids), C.c_void_p(got.ptr), 1, None, None)
    for k, dt in enumerate(DTS):
        p = C.byref(b._phys())
        L.call("gs_clock_set_dt", C.c_void_p(b._clock.ptr), C.c_double(dt), p, b._fo.s, None)
        L.call("gs_flat_step", C.byref(b._desc()), p, b._fo.s, C.c_void_p(b._clock.ptr), None)
        L.call("gs_flat_sample", C.byref(b._desc()), C.c_void_p(b._clock.ptr), C.c_void_p(d_ids.ptr), len(ids),
               C.c_void_p(want.ptr + k * len(ids) * es), None)
    L.sync(None)
    assert np.array_equal(a.q_flat(), b.q_flat())
    assert np.array_equal(got.download(), want.download())
