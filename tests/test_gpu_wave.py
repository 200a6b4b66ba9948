"""The wavefront forms on the GPU: the root and the quotient over every input within their
bounds, and sweeps whose rows leave those bounds (they go to the general functions row by
row) against the oracle, at the edges of the sweep's tiles."""
import numpy as np
import pytest

from geoswe_amd import Config, Mesh2D, Solver2D
from oracle import swe_oracle as O

pytestmark = pytest.mark.gpu


def test_wave_root_and_quotient_equal_ieee(gpu):
    from geoswe_amd import _lib as L
    counts = L.DeviceArray((4,), np.uint64, zero=True)
    L.call("gs_crmath_check", 4, counts.ptr, None)
    L.sync(None)
    c = counts.download()
    assert c[0] == 0, f"root: {int(c[0])} mismatches, last input {int(c[1]) - 1:#x}"
    assert c[2] == 0, f"quotient: {int(c[2])} mismatches, last index {int(c[3]) - 1:#x}"


def _oracle_residual(q0, bed, dx, bc):
    g = 4
    nx, ny = bed.shape
    qp = np.zeros((3, nx + 2 * g, ny + 2 * g), np.float32)
    qp[:, g:-g, g:-g] = q0
    O.bc_fill(qp, g, *bc)
    bp = O.pad_bed(bed, g, *bc, dtype=np.float32)
    return O.residual(qp, bp, dx, dx, 9.81, 1e-6)[:, g:-g, g:-g]


def _state(nx, ny, odd):
    rng = np.random.default_rng(nx * 1000 + ny)
    bed = (rng.random((nx, ny)) * 1.2).astype(np.float32)
    h = np.maximum(0.8 - bed, 0.0).astype(np.float32)
    q = np.stack([h, (rng.random((nx, ny)) - 0.5).astype(np.float32) * h,
                  (rng.random((nx, ny)) - 0.5).astype(np.float32) * h]).astype(np.float32)
    if odd:   # finite operands that the short forms do not take, in a few cells
        i = rng.integers(0, nx, 6)
        j = rng.integers(0, ny, 6)
        q[0, i, j] = 0.5
        q[1, i[0], j[0]] = 4.0e3          # a velocity of 8000 m/s
        q[1, i[1], j[1]] = 1.0e-30        # momenta too small for an exact remainder
        q[2, i[2], j[2]] = -1.0e-42
        q[0, i[3], j[3]] = 1.0e-33        # a film whose root is in the general range
        bed[i[4], j[4]] = 3.0e6
        q[0, i[5], j[5]] = 2.0e6
    return q, bed


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("shape,rows", [((4, 4), 0), ((7, 59), 1), ((13, 60), 2), ((9, 61), 3), ((33, 123), 5),
                                        ((40, 600), 1 << 20)])
@pytest.mark.parametrize("bc", [("wall", "periodic"), ("fall", "extrapolate")])
def test_residual_and_steps_at_tile_edges(gpu, shape, rows, bc, odd):
    """The residual is the oracle's bit for bit, and two steps give the same bits at every tile
    height (1 << 20 rows takes the sweep with 64-bit offsets), also in rows left to the general
    functions."""
    nx, ny = shape
    q, bed = _state(nx, ny, odd)

    def solver(tile_rows):
        cfg = Config(bc_x=bc[0], bc_y=bc[1], dtype="float32", friction="manning", manning_n=0.03)
        return Solver2D(Mesh2D(nx, ny, 2.0, 2.0, ngh=4), cfg, q, bed, tile_rows=tile_rows)

    s = solver(rows)
    got = s.residual()
    want = _oracle_residual(q, bed, 2.0, bc)
    assert np.array_equal(got, want)
    ref = solver(64)
    for dt in (1e-3, 2e-3):
        s.step(dt)
        ref.step(dt)
    assert np.array_equal(s.q_interior, ref.q_interior)
    assert s._clockv().lam_bits == ref._clockv().lam_bits


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("ext,maxh", [(False, False), (False, True), (True, True)])
@pytest.mark.parametrize("shape,rows", [((6, 5), 1), ((17, 61), 2), ((33, 124), 5), ((40, 130), 2000)])
def test_flat_sweep_at_tile_edges(gpu, shape, rows, ext, maxh, dtype, odd):
    """Three steps of the flat sweep (lean, plain and extended) give the chunk traversal's bits, at
    tiles of one row and more, cut by an irregular mask, and a height (2000) that the wavefront
    forms leave to the general functions whole; in rows with odd operands too."""
    from geoswe_amd import CompressedSolver
    nx, ny = shape
    q, bed = _state(nx, ny, odd)
    if odd and dtype == "float64":
        q, bed = q.astype(np.float64), bed.astype(np.float64)
        q[1, nx // 2, ny // 2] = 1.0e-300
    rng = np.random.default_rng(nx + ny)
    mask = rng.random((nx, ny)) > 0.06
    mask[nx // 2, ny // 2] = True
    cls = rng.integers(0, 3, (nx, ny)).astype(np.uint8)
    out = []
    for trav in ("tiles", "chunks"):
        cfg = Config(bc_x="fall", bc_y="fall", dtype=dtype, friction="manning", manning_n=0.03,
                     rainfall=20.0 / 3.6e6)
        s = Solver2D(Mesh2D(nx, ny, 2.0, 2.0), cfg, q.astype(dtype), bed.astype(dtype))
        s.set_inside_mask(mask)
        c = CompressedSolver.from_dense(s, cfl_linf=True, track_max_depth=maxh, sweep_rows=rows)
        if ext:
            g = s.mesh.ngh
            c.set_ga_drain({"cls_pad": np.pad(cls, g), "Ks_t": [0.0, 1e-5, 4e-5], "psi_t": [0.1, 0.1, 0.2],
                            "dth_t": [0.3, 0.3, 0.3], "F_pad": None,
                            "inv_tau_pad": np.full((nx + 2 * g, ny + 2 * g), 1.0 / 600.0), "mode": "fused"})
        c.traversal = trav
        c.advance(3)
        out.append((c.q_flat(), c.t, c.nsteps, c.max_depth() if maxh else None))
    a, b = out
    assert a[1:3] == b[1:3] and np.array_equal(a[0], b[0])
    assert not maxh or np.array_equal(a[3], b[3])


@pytest.mark.parametrize("dtype,compute", [("float32", None), ("float64", None), ("float32", "float64")])
@pytest.mark.parametrize("manning", ["flags", "plane", "field"])
@pytest.mark.parametrize("gridded,masked", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("shape,rows", [((5, 61), 1), ((23, 130), 4)])
def test_dense_planes_loaded_ahead(gpu, shape, rows, gridded, masked, manning, dtype, compute):
    """The cells' flags, classes, Manning field, rain frame and running maximum loaded a row ahead give
    the bits of the sweep with 64-bit offsets (tile height 1 << 20), which loads them at their use."""
    from geoswe_amd import RainfallForcing, StageBoundary
    nx, ny = shape
    rng = np.random.default_rng(nx + ny)
    q, bed = _state(nx, ny, False)
    mask = rng.random((nx, ny)) > 0.1
    frames = rng.random((2, nx, ny)) * 4.0e4
    cls = rng.integers(0, 40 if manning == "plane" else 5, (nx, ny)).astype(np.uint8)
    n_of = np.linspace(0.02, 0.09, 40 if manning == "plane" else 5)
    mesh = Mesh2D(nx, ny, 2.0, 2.0, ngh=4)
    sea = np.zeros((nx, ny), bool)
    sea[:, 0] = True
    out = []
    for tile_rows in (rows, 1 << 20):
        kw = dict(rainfall_forcing=RainfallForcing(np.array([0.0, 2e-3]), frames)) if gridded else \
            dict(rainfall=20.0 / 3.6e6)
        if masked:
            kw["stage_boundary"] = StageBoundary.from_mask(sea, mesh, bed, np.array([0.0, 1.0]), np.array([0.9, 1.4]))
        cfg = Config(bc_x="fall", bc_y="wall", dtype=dtype, compute_dtype=compute, friction="manning",
                     manning_n=0.03, **kw)
        s = Solver2D(mesh, cfg, q.astype(dtype), bed.astype(dtype), tile_rows=tile_rows)
        if manning == "field":
            s.set_manning(n_of[cls] + 1e-3 * np.arange(ny))
        else:
            s.set_manning_table(np.pad(cls, 4, mode="edge"), n_of)
        if masked:
            s.set_inside_mask(mask)
            s.set_cfl_ghost_mask(~mask)
        for dt in (1e-3, 2e-3, 1e-3):
            s.step(dt)
        out.append((s.q_interior, s.max_depth(), s._clockv().lam_bits))
    a, b = out
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]
