"""The work that users of geoswe_amd have it do, as cases that can be timed and compared.

Every case goes through the package's own entry points: ``Solver2D`` (run, advance, captured
steps) on the dense grid, ``CompressedSolver`` on the active cells of a coastal domain,
``Ensemble`` over many domains, and the torch autograd function of the gauge misfit. The
fields (beds, land cover, rain) are made on the GPU with torch from the seed alone.

``exact`` steps the same inputs in float64 with plain torch operations: the HLLC flux with
surface reconstruction, rain, point-implicit Manning friction, the wet/dry rule and the CFL
time step, written out below without the package.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

G = 9.81
H_MIN = 1.0e-6        # dry floor of every case, in either precision
CFL = 0.5
VCAP = 15.0           # the friction velocity cap of Config
NGH = 4               # ghost layers of Mesh2D
TIDE_S = 44712.0      # M2 tide
N_CLASSES = 8
FLOPS_STEP = 230.0    # arithmetic of one cell update: two faces, their sums, friction, wave speed


def listed() -> list:
    return [
        # the first thing a user runs: a small dam break stepped to the next output time and read
        # back for a plot; launches, the clock's reads and the host loop are most of it
        dict(name="frames_dam_break_256", kind="frames", nx=256, ny=256, bc="wall", frame_s=1.0),
        # a small catchment inside a larger program, its steps captured once in a HIP graph
        dict(name="graph_500x517", kind="dense", nx=500, ny=517, dtype="float32", arith="float32", mode="graph",
             steps=20),
        # the one-million-cell and 16.8-million-cell grids that dense solvers are quoted on
        dict(name="dense_1m", kind="dense", nx=1024, ny=1024, dtype="float32", arith="float32", mode="advance",
             steps=20),
        dict(name="dense_16m", kind="dense", nx=4096, ny=4096, dtype="float32", arith="float32", mode="advance",
             steps=10),
        # the headline grid: rain on a slope, 640 M cells, everywhere wet
        dict(name="dense_640m", kind="dense", nx=25600, ny=25000, dtype="float32", arith="float32", mode="advance",
             steps=2),
        # double precision, for reference runs
        dict(name="dense_f64_1537x2111", kind="dense", nx=1537, ny=2111, dtype="float64", arith="float64",
             mode="advance", steps=6),
        # float32 storage with float64 arithmetic: long runs whose round-off has to stay small
        dict(name="dense_mixed_1999x2003", kind="dense", nx=1999, ny=2003, dtype="float32", arith="float64",
             mode="advance", steps=6),
        # a coastal city on its active cells: land cover classes, gridded rain, a tide at the edge
        dict(name="coastal_flat_2048", kind="coastal", n=2048, layout="flat", dtype="float32", tail=False, maxh=False,
             steps=20),
        # the same with an operational driver's whole tail of forcings and the running maximum depth
        dict(name="coastal_forced_1500", kind="coastal", n=1500, layout="flat", dtype="float32", tail=True, maxh=True,
             steps=10),
        # the masked dense form of a coastal domain, with its running maximum depth
        dict(name="coastal_dense_1021", kind="coastal", n=1021, layout="dense", dtype="float32", tail=False, maxh=True,
             steps=10),
        # an ensemble forecast: sixteen uneven members stepped together
        dict(name="ensemble_16", kind="ensemble", members=16, lo=256, hi=1024, steps=20),
        # calibration of Manning's n and the bed against gauges: a loss and its gradient
        dict(name="adjoint_1536", kind="adjoint", n=1536, steps=40, every=20),
    ]


def draw(rng: random.Random) -> dict:
    """One more case of the same ranges."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["frames", "dense", "dense", "dense", "coastal", "coastal", "ensemble", "adjoint"])
    if kind == "frames":
        nx = log_int(48, 700)
        return dict(kind=kind, nx=nx, ny=max(40, int(nx * rng.uniform(0.5, 2.0))),
                    bc=rng.choice(["wall", "periodic", "extrapolate"]), frame_s=round(rng.uniform(0.3, 2.0), 3))
    if kind == "dense":
        cells = log_int(6.0e4, 6.4e8)
        dtype, arith = rng.choice([("float32", "float32")] * 4 + [("float64", "float64"), ("float32", "float64")])
        if arith == "float64":
            cells = min(cells, log_int(6.0e4, 3.0e7))
        aspect = rng.uniform(0.5, 2.0)
        nx = max(40, int(math.sqrt(cells * aspect)))
        ny = max(40, int(cells / nx))
        mode = "graph" if cells < 4.0e6 and rng.random() < 0.3 else "advance"
        return dict(kind=kind, nx=nx, ny=ny, dtype=dtype, arith=arith, mode=mode,
                    steps=2 if cells > 1.0e8 else 2 * rng.randint(2, 10))
    if kind == "coastal":
        n = log_int(150, 2600)
        layout = rng.choice(["flat", "flat", "dense"])
        dtype = rng.choice(["float32"] * 4 + ["float64"])
        tail = layout == "flat" and rng.random() < 0.3
        return dict(kind=kind, n=n, layout=layout, dtype=dtype, tail=tail, maxh=rng.random() < 0.5,
                    steps=2 * rng.randint(2, 10))
    if kind == "ensemble":
        return dict(kind=kind, members=rng.randint(3, 16), lo=log_int(128, 300), hi=log_int(400, 1200),
                    steps=2 * rng.randint(5, 15))
    return dict(kind=kind, n=log_int(128, 1800), steps=2 * rng.randint(8, 25), every=rng.randint(8, 25))


# --------------------------------------------------------------------------- fields
def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    return g


def _fractal(nx: int, ny: int, seed: int, longest: float = 1024.0, hurst: float = 0.8, octaves: int = 6,
             dtype=torch.float32) -> torch.Tensor:
    """A rough (nx, ny) field in [-1, 1]: octaves of smooth noise whose amplitude falls with their
    wavelength (in cells) to the power `hurst`."""
    gen = _gen(seed)
    out = torch.zeros((nx, ny), dtype=dtype, device="cuda")
    wave, amp, total = float(longest), 1.0, 0.0
    for _ in range(octaves):
        if wave < 3.0:
            break
        sx, sy = max(3, int(nx / wave) + 2), max(3, int(ny / wave) + 2)
        coarse = torch.rand((1, 1, sx, sy), generator=gen, device="cuda", dtype=torch.float32).to(dtype) * 2.0 - 1.0
        fine = torch.nn.functional.interpolate(coarse, size=(nx, ny), mode="bilinear", align_corners=True)[0, 0]
        out.add_(fine, alpha=amp)
        total += amp
        wave, amp = wave / 4.0, amp * 4.0 ** (-hurst)
    return out.div_(total)


class _Plane:
    """A device array of the package as torch sees one."""

    def __init__(self, arr, shape):
        self.arr = arr
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": np.dtype(arr.dtype).str,
                                         "data": (arr.ptr, False), "version": 2}


def _view(arr, shape=None) -> torch.Tensor:
    return torch.as_tensor(_Plane(arr, shape or arr.shape), device="cuda")


class _Raw:
    """A raw device plane (pointer, shape, dtype) as torch sees one."""

    def __init__(self, ptr, shape, dtype):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": np.dtype(dtype).str, "data": (ptr, False),
                                         "version": 2}


# --------------------------------------------------------------------------- dense cases
def _dam_break(case: dict, seed: int):
    """(h, bed) of a circular dam break: still water inside a seeded disc over shallow water."""
    nx, ny = case["nx"], case["ny"]
    rng = np.random.default_rng(seed)
    r = 0.16 * min(nx, ny) * rng.uniform(0.9, 1.1)
    ci, cj = nx * rng.uniform(0.45, 0.55), ny * rng.uniform(0.45, 0.55)
    i, j = np.arange(nx)[:, None], np.arange(ny)[None, :]
    h = np.where(np.hypot(i - ci, j - cj) < r, rng.uniform(8.0, 12.0), 1.0)
    return h, np.zeros((nx, ny))


SLOPE_DX, SLOPE_N, SLOPE_RAIN, SLOPE_H0 = 3.0, 0.03, 50.0 / 3.6e6, 0.1
SLOPE_WARM = 10       # steps before the timed ones, so that water runs down the slope


def _slope_bed(case: dict, seed: int) -> torch.Tensor:
    """A planar 1e-3 slope with half a metre of fractal relief, in the state's precision."""
    nx, ny = case["nx"], case["ny"]
    dt = torch.float64 if case["dtype"] == "float64" else torch.float32
    b = _fractal(nx, ny, seed, dtype=dt).mul_(0.5)
    return b.add_(torch.arange(nx, device="cuda", dtype=dt)[:, None] * (1.0e-3 * SLOPE_DX))


def _slope_solver(case: dict, seed: int):
    from geoswe_amd import Config, Mesh2D, Solver2D
    nx, ny = case["nx"], case["ny"]
    cfg = Config(bc_x="fall", bc_y="fall", cfl=CFL, dtype=case["dtype"], friction="manning", manning_n=SLOPE_N,
                 rainfall=SLOPE_RAIN, h_min=H_MIN, h_min_cfl=H_MIN,
                 compute_dtype="float64" if case["arith"] == "float64" else None)

    def write(ptr, pitch, _code):
        plane = torch.as_tensor(_Raw(ptr, (nx, pitch), case["dtype"]), device="cuda")
        plane[:, :ny] = _slope_bed(case, seed)
        torch.cuda.synchronize()

    return Solver2D(Mesh2D(nx, ny, SLOPE_DX, SLOPE_DX, ngh=NGH), cfg, None, None, track_max_depth=False,
                    device_init=(SLOPE_H0, write))


# --------------------------------------------------------------------------- coastal cases
def _spread(mask: torch.Tensor, steps: int) -> torch.Tensor:
    """`steps` dilations by the 4-neighbour cross."""
    m = mask.clone()
    for _ in range(steps):
        o = m.clone()
        o[1:] |= m[:-1]
        o[:-1] |= m[1:]
        o[:, 1:] |= m[:, :-1]
        o[:, :-1] |= m[:, 1:]
        m = o
    return m


COAST_DX = 3.0
COAST_WARM = 10


def _coast_fields(n: int, seed: int, dtype: str) -> dict:
    """A coastal domain as host arrays: land above -2 m plus a nearshore band (~45 % of the box) is
    active; eight Manning classes in patches; rain of 0-80 mm/h in three frames; a tide on the
    active sea edge; still water at sea level and a flood standing on part of the land. The
    terrain goes with the size and a few centimetres of survey error with the seed, so that the
    active set is the same for every scenario run on a domain."""
    rng = np.random.default_rng(seed)
    raw = _fractal(n, n, n, longest=max(64.0, n / 4.0))
    thr = torch.quantile(raw[:: max(1, n // 512), :: max(1, n // 512)].reshape(-1)[:1_000_000], 0.6)
    lo, hi = raw.min(), raw.max()
    bed = torch.where(raw < thr, -2.0 + (raw - thr) * (8.0 / (thr - lo)), -2.0 + (raw - thr) * (62.0 / (hi - thr)))
    active = _spread(bed > -2.0, max(4, n // 128))
    edge = torch.zeros_like(active)
    edge[0, :] = edge[-1, :] = edge[:, 0] = edge[:, -1] = True
    sea = edge & active & (bed < -2.1)
    bed += 0.05 * _fractal(n, n, seed, longest=64.0, octaves=3)
    sites = 48
    ii = torch.arange(n, device="cuda", dtype=torch.float32)[:, None]
    jj = torch.arange(n, device="cuda", dtype=torch.float32)[None, :]
    near = torch.full((n, n), math.inf, device="cuda")
    cls = torch.zeros((n, n), dtype=torch.uint8, device="cuda")
    for x, y, c in zip(rng.uniform(0, n, sites), rng.uniform(0, n, sites), rng.integers(0, N_CLASSES, sites)):
        d = (ii - float(x)) ** 2 + (jj - float(y)) ** 2
        cls = torch.where(d < near, torch.full_like(cls, int(c)), cls)
        near = torch.minimum(near, d)
    rain = []
    for k in range(3):
        f = _fractal(n, n, seed + 1000 + k, longest=max(32.0, n / 2.0), octaves=3)
        rain.append(((f - f.min()) * (80.0 / (f.max() - f.min()))).cpu().numpy())
    b = bed.cpu().numpy()
    act = active.cpu().numpy()
    flood = _fractal(n, n, seed + 77, longest=max(32.0, n / 8.0), octaves=3).cpu().numpy()
    h = np.maximum(-b, 0.0)
    h = np.where((b >= 0.0) & act & (flood > 0.1), 2.0 * flood.clip(0.0, 1.0), h).astype(dtype)
    ts = np.linspace(0.0, 2.0 * TIDE_S, 401)
    return dict(n=n, bed=b.astype(dtype), h=h, active=act, cls=cls.cpu().numpy(),
                rain=np.stack(rain).astype(np.float32) * np.float32(rng.uniform(0.5, 1.5)),
                rain_t=np.arange(3) * 300.0, ntab=np.linspace(0.02, 0.12, N_CLASSES) * rng.uniform(0.8, 1.2, N_CLASSES),
                sea=sea.cpu().numpy(), tide_t=ts, tide=0.8 + np.sin(2.0 * np.pi * ts / TIDE_S))


def _coast_case(f: dict, dtype: str):
    """The package's own description of such a domain."""
    from geoswe_amd import Config, Mesh2D, RainfallForcing, StageBoundary
    from geoswe_amd.cases import CoastalCase
    mesh = Mesh2D(f["n"], f["n"], COAST_DX, COAST_DX, ngh=NGH)
    stage = StageBoundary.from_mask(f["sea"], mesh, f["bed"], f["tide_t"], f["tide"]) if f["sea"].any() else None
    cfg = Config(bc_x="fall", bc_y="fall", cfl=CFL, dtype=dtype, friction="manning", h_min=H_MIN, h_min_cfl=H_MIN,
                 rainfall_forcing=RainfallForcing(time_s=f["rain_t"], rate_mm_h=f["rain"]), stage_boundary=stage)
    q0 = np.stack([f["h"], np.zeros_like(f["h"]), np.zeros_like(f["h"])])
    return CoastalCase(mesh=mesh, cfg=cfg, q0=q0, bed=f["bed"], active=f["active"], cls=f["cls"],
                       ntab=f["ntab"].astype(np.float32), sea_edge=f["sea"])


def _sides(case: dict) -> list:
    """The members' sides, spread over the logarithm of their range."""
    m, lo, hi = case["members"], case["lo"], case["hi"]
    return [int(round(lo * (hi / lo) ** (((k * 7) % m) / max(1, m - 1)))) for k in range(m)]


GAUGES = 32
ADJ_WARM = 10


# --------------------------------------------------------------------------- prepare, run
def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "frames":
        from geoswe_amd import Config, Mesh2D, Solver2D
        h, b = _dam_break(case, seed)
        cfg = Config(bc_x=case["bc"], bc_y=case["bc"], cfl=CFL, dtype="float32", h_min=H_MIN, h_min_cfl=H_MIN)
        s = Solver2D(Mesh2D(case["nx"], case["ny"], 1.0, 1.0, ngh=NGH), cfg, np.stack([h, 0 * h, 0 * h]), b)
        return dict(kind=kind, solver=s, t=0.0, frame=case["frame_s"])
    if kind == "dense":
        s = _slope_solver(case, seed)
        s.advance(SLOPE_WARM)
        st = dict(kind=kind, solver=s, steps=case["steps"], graph=None)
        if case["mode"] == "graph":
            st["graph"] = s.capture_steps(case["steps"])
        # an even number of steps leaves the state in the first of the two buffers
        st["out"] = [_view(s._bufs[0][k])[:, :case["ny"]] for k in range(3)]
        return st
    if kind == "coastal":
        c = _coast_case(_coast_fields(case["n"], seed, case["dtype"]), case["dtype"])
        if case["layout"] == "dense":
            s = c.dense(track_max_depth=case["maxh"])
            out = [_view(s._bufs[0][k])[:, :case["n"]] for k in range(3)]
            if case["maxh"]:
                out.append(_view(s._max_h)[:, :case["n"]])
        else:
            s = c.flat(track_max_depth=case["maxh"])
            if case["tail"]:
                from geoswe_amd.cases import attach_coastal_forcings
                attach_coastal_forcings(c, s, band=max(4, case["n"] // 64), n_clamp=case["n"], n_drain=case["n"] // 2,
                                        seed=seed)
            out = [_view(s._bufs[0][k]) for k in range(3)]
            if case["maxh"]:
                out.append(_view(s._max_h))
            if case["tail"]:
                out.append(_view(s._ga["F"]))
        s.advance(COAST_WARM)
        return dict(kind=kind, solver=s, steps=case["steps"], out=out, graph=None)
    if kind == "ensemble":
        from geoswe_amd.ensemble import Ensemble
        members = [_coast_case(_coast_fields(n, seed + 31 * k, "float32"), "float32").flat()
                   for k, n in enumerate(_sides(case))]
        e = Ensemble(members, graph_batch=10)
        e.advance(COAST_WARM)
        return dict(kind=kind, ens=e, steps=case["steps"], out=[_view(m._bufs[0][k]) for m in members for k in range(3)])
    from geoswe_amd.adjoint import GaugeMisfit
    f = _coast_fields(case["n"], seed, "float32")
    c = _coast_case(f, "float32")
    ref = c.flat()
    dts = np.array([ref.step() for _ in range(case["steps"])])
    s = c.flat()
    prob = GaugeMisfit(s, _gauge_ids(s.fm.active, s.q_flat()[0], seed), dts, checkpoint_every=case["every"])
    ntab, bed = prob.params()
    prob.set_params(ntab=ntab * _truth(seed))       # the run that the gauges recorded
    prob.h_star = prob.simulate(keep_checkpoints=False).copy()
    prob.set_params(ntab=ntab)
    return dict(kind=kind, prob=prob, ntab=torch.tensor(ntab, dtype=torch.float32, device="cuda"),
                bed=torch.tensor(bed, dtype=torch.float32, device="cuda"))


def _gauge_ids(active: np.ndarray, h: np.ndarray, seed: int) -> np.ndarray:
    wet = np.flatnonzero(active & (h > 0.05))
    return np.sort(np.random.default_rng(seed + 5).choice(wet, size=min(GAUGES, len(wet)), replace=False))


def _truth(seed: int) -> np.ndarray:
    return 1.0 + 0.25 * np.random.default_rng(seed + 6).uniform(-1.0, 1.0, N_CLASSES)


def run(state: dict):
    kind = state["kind"]
    if kind == "frames":
        state["t"] += state["frame"]
        state["solver"].run(state["t"])
        return state["solver"].q_interior
    if kind in ("dense", "coastal"):
        if state["graph"] is not None:
            state["graph"].replay()
            state["solver"].sync()
        else:
            state["solver"].advance(state["steps"])
        return state["out"]
    if kind == "ensemble":
        state["ens"].advance(state["steps"])
        return state["out"]
    from geoswe_amd.adjoint import GaugeMisfitFn
    n = state["ntab"].clone().requires_grad_(True)
    b = state["bed"].clone().requires_grad_(True)
    loss = GaugeMisfitFn.apply(n, b, state["prob"])
    loss.backward()
    return {"loss": loss.detach(), "n": n.grad, "bed": b.grad}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "frames":
        # about 9 m/s of wave speed on 1 m cells; the state in and out and the bed, then the read-back
        steps = max(1.0, case["frame_s"] * 18.0)
        cells = case["nx"] * case["ny"]
        return {"bytes": cells * (28.0 * steps + 12.0), "flops": FLOPS_STEP * cells * steps}
    if kind == "dense":
        cells = case["nx"] * case["ny"] * case["steps"]
        return {"bytes": cells * (56.0 if case["dtype"] == "float64" else 28.0), "flops": FLOPS_STEP * cells}
    if kind == "coastal":
        # state in and out, bed and rain in the state's type, a byte of class and flags
        cells = 0.45 * case["n"] ** 2 * case["steps"]
        es = 8 if case["dtype"] == "float64" else 4
        per = 8 * es + 1 + (es if case["maxh"] else 0) + (4 * es + 1 if case["tail"] else 0)
        return {"bytes": cells * per, "flops": (FLOPS_STEP + (30.0 if case["tail"] else 0.0)) * cells}
    if kind == "ensemble":
        cells = 0.45 * sum(n * n for n in _sides(case)) * case["steps"]
        return {"bytes": cells * 33.0, "flops": FLOPS_STEP * cells}
    # two forward passes (the second from checkpoints, keeping what the reverse reads) and the reverse
    cells = 0.45 * case["n"] ** 2 * case["steps"]
    return {"bytes": cells * (33.0 + 45.0 + 72.0), "flops": cells * (2.0 * FLOPS_STEP + 600.0)}


# --------------------------------------------------------------------------- float64 values
def _sel(m, a, b):
    return torch.where(m, a, b)


def _root(x):
    ok = x > 0
    return _sel(ok, torch.sqrt(_sel(ok, x, torch.ones_like(x))), torch.zeros_like(x))


def _quot(a, b, ok):
    return _sel(ok, a / _sel(ok, b, torch.ones_like(b)), torch.zeros_like(a))


def _up(x):                       # max(x, 0), with no slope at 0
    return _sel(x > 0, x, torch.zeros_like(x))


def _lo(a, b):
    return _sel(a <= b, a, b)


def _hi(a, b):
    return _sel(a >= b, a, b)


def _face64(bL, bR, gzL, gzR, hL, hR, nL, tL, nR, tR, half):
    """Fluxes (mass, normal, transverse) and the bed sources of both cells at faces between L and R,
    zero where both cells are dry; elevations are relative to the bed of L."""
    db = bR - bL
    zL = half * gzL
    zR = db - half * gzR
    zf = _up(db)
    dzc = zR - zL
    dz = db - dzc
    eR = hR + db
    dryl, dryr = hL < H_MIN, hR < H_MIN
    fl = _up(hL + _up(_lo(dz, eR - hL)) - zf)
    fr = _up(eR + _up(_lo(-dz, hL - eR)) - zf)
    headl, headr = zf - hL, zf - eR
    sL = 0.5 * G * (fl + hL) * (zf - _sel(dryr, _up(headl), _up(_lo(dzc, headl))))
    sR = 0.5 * G * (fr + hR) * (zf - _sel(dryl, _up(headr), _up(_lo(-dzc, headr))) - db)
    # HLLC
    cl, cr = _root(G * fl), _root(G * fr)
    us = 0.5 * (nL + nR) + cl - cr
    cs = _up(0.5 * (cl + cr) + 0.25 * (nL - nR))
    d1, d2 = fl <= H_MIN, fr <= H_MIN
    zero = torch.zeros_like(fl)
    SL = _sel(d1, nR - 2.0 * cr, _lo(nL - cl, us - cs))
    SR = _sel(d2, nL + 2.0 * cl, _hi(nR + cr, us + cs))
    SL, SR = _sel(d1 & d2, zero, SL), _sel(d1 & d2, zero, SR)
    den = fr * (nR - SR) - fl * (nL - SL)
    big = den.abs() > 1.0e-14
    SM = _sel(big, _quot(SL * fr * (nR - SR) - SR * fl * (nL - SL), den, big), 0.5 * (nL + nR))
    left, right = SL >= 0, ~(SM >= 0) & ~(SR >= 0)
    one = left | right
    lft = _sel(one, left, SM >= 0)
    S, n, t, h = _sel(lft, SL, SR), _sel(lft, nL, nR), _sel(lft, tL, tR), _sel(lft, fl, fr)
    hs = h * _quot(S - n, (S - SM) + 1.0e-30, ~one)
    F = h * n
    M = F * n + 0.5 * G * h * h
    T = F * t
    F2, M2, T2 = F + S * (hs - h), M + S * (hs * SM - F), T + S * (hs * t - h * t)
    wet = ~(dryl & dryr)
    return tuple(_sel(wet, x, zero) for x in (_sel(one, F, F2), _sel(one, M, M2), _sel(one, T, T2), sL, sR))


def _step64(q, b, n, rain, dt, upd, d, friction, stage=None, eta=0.0):
    """One step of the cells marked `upd` (never in the two outermost rows and columns)."""
    h, hu, hv = q[0], q[1], q[2]
    wet = h > H_MIN
    u, v = _quot(hu, h, wet), _quot(hv, h, wet)
    pad = torch.nn.functional.pad
    gx = pad((0.5 / d) * (b[2:] - b[:-2]), (0, 0, 1, 1))
    gy = pad((0.5 / d) * (b[:, 2:] - b[:, :-2]), (1, 1))
    X = _face64(b[:-1], b[1:], gx[:-1], gx[1:], h[:-1], h[1:], u[:-1], v[:-1], u[1:], v[1:], 0.5 * d)
    Y = _face64(b[:, :-1], b[:, 1:], gy[:, :-1], gy[:, 1:], h[:, :-1], h[:, 1:], v[:, :-1], u[:, :-1], v[:, 1:],
                u[:, 1:], 0.5 * d)
    xp, xm = [pad(a, (0, 0, 0, 1)) for a in X], [pad(a, (0, 0, 1, 0)) for a in X]
    yp, ym = [pad(a, (0, 1)) for a in Y], [pad(a, (1, 0)) for a in Y]
    r0 = (xm[0] - xp[0] + ym[0] - yp[0]) / d
    r1 = (xm[1] - xp[1] - xp[3] + xm[4] + ym[2] - yp[2]) / d
    r2 = (xm[2] - xp[2] + ym[1] - yp[1] - yp[3] + ym[4]) / d
    h1, a, c = h + dt * (r0 + rain), hu + dt * r1, hv + dt * r2
    dry = h1 < H_MIN
    if friction:
        hs = _sel(dry, torch.ones_like(h1), h1)
        speed = _root((a / hs) ** 2 + (c / hs) ** 2)
        w = hs ** (-4.0 / 3.0)
        ncri = _root(1.0 / ((1.0e-10 + dt) * G * w * (speed + 1.0e-30)))
        nn = _sel((speed > VCAP) & (ncri > n), ncri, n + torch.zeros_like(h1))
        k = 2.0 / (torch.sqrt(1.0 + 4.0 * dt * G * nn * nn * w * speed) + 1.0)
        a, c = a * k, c * k
    zero = torch.zeros_like(h1)
    h1, a, c = _sel(dry, _up(h1), h1), _sel(dry, zero, a), _sel(dry, zero, c)
    if stage is not None:
        h1, a, c = _sel(stage, _up(eta - b), h1), _sel(stage, zero, a), _sel(stage, zero, c)
    return _sel(upd[None], torch.stack([h1, a, c]), q)


def _dt64(q, upd, d):
    h = q[0]
    ok = upd & (h >= H_MIN)
    hs = _sel(ok, h, torch.ones_like(h))
    lam = _sel(ok, torch.maximum(q[1].abs(), q[2].abs()) / hs + torch.sqrt(G * hs), torch.zeros_like(h)).max()
    return CFL * d / (max(float(lam), math.sqrt(G * H_MIN)) + 1.0e-12)


def _ghosts(q, kind):
    """Two ghost layers on every side of a padded state, x then y."""
    for ax in (1, 2):
        q = q.transpose(1, ax)
        if kind == "fall":
            q[:, :2] = 0.0
            q[:, -2:] = 0.0
        elif kind == "periodic":
            q[:, :2], q[:, -2:] = q[:, -4:-2].clone(), q[:, 2:4].clone()
        elif kind == "extrapolate":
            q[:, :2], q[:, -2:] = q[:, 2:3].clone(), q[:, -3:-2].clone()
        else:
            q[:, :2], q[:, -2:] = q[:, 2:4].flip(1).clone(), q[:, -4:-2].flip(1).clone()
            q[ax, :2] *= -1.0
            q[ax, -2:] *= -1.0
        q = q.transpose(1, ax)
    return q


def _pad_bed(b, k, kind):
    mode = "circular" if kind == "periodic" else "replicate"
    return torch.nn.functional.pad(b[None, None], (k, k, k, k), mode=mode)[0, 0]


def _dense64(h, b, d, kind, n, rain, friction, steps=None, t_end=None):
    b = _pad_bed(b, 2, kind)
    q = torch.zeros((3, *b.shape), dtype=torch.float64, device="cuda")
    q[0, 2:-2, 2:-2] = h
    upd = torch.zeros(b.shape, dtype=torch.bool, device="cuda")
    upd[2:-2, 2:-2] = True
    t, k = 0.0, 0
    while (k < steps) if steps is not None else (t < t_end - 1.0e-12):
        q = _ghosts(q, kind)
        dt = _dt64(q, upd, d)
        if t_end is not None and t + dt > t_end:
            dt = t_end - t
        q = _step64(q, b, n, rain, dt, upd, d, friction)
        t, k = t + dt, k + 1
    return q[:, 2:-2, 2:-2]


class _Coast64:
    """A coastal domain on its padded box: inactive cells keep their value."""

    def __init__(self, f: dict, dtype: str):
        n, k = f["n"], NGH
        dev = lambda x: torch.as_tensor(np.ascontiguousarray(x), device="cuda")
        grow = lambda x: torch.nn.functional.pad(x, (k, k, k, k))
        self.n = n
        self.b = _pad_bed(dev(f["bed"]).double(), k, "fall")
        self.q = torch.zeros((3, n + 2 * k, n + 2 * k), dtype=torch.float64, device="cuda")
        self.q[0, k:-k, k:-k] = dev(f["h"]).double()
        self.act = grow(dev(f["active"]))
        self.sea = grow(dev(f["sea"]))
        self.cls = grow(dev(f["cls"]).long())
        self.ntab = dev(f["ntab"].astype(np.float32)).double()
        self.rain = [grow(dev((r / 3.6e6).astype(dtype)).double()) for r in f["rain"]]
        self.f = f
        # stored cells: the active ones and two rings around them, row by row
        self.stored = _spread(self.act, 2)

    def eta(self, t):
        return float(np.interp(t, self.f["tide_t"], self.f["tide"]))

    def step(self, q, b, ntab, t, dt):
        k = int(np.searchsorted(self.f["rain_t"], t, side="right")) - 1
        return _step64(q, b, ntab[self.cls], self.rain[min(max(k, 0), 2)], dt, self.act, COAST_DX, True, self.sea,
                       self.eta(t + dt))

    def run(self, steps, max_from=None):
        q, t = self.q, 0.0
        top = torch.zeros_like(q[0])
        for _ in range(steps):
            dt = _dt64(q, self.act, COAST_DX)
            q = self.step(q, self.b, self.ntab, t, dt)
            t += dt
            top = _sel(self.act, torch.maximum(top, q[0]), top)
        return q, top


def exact(case: dict, seed: int):
    kind = case["kind"]
    dev = lambda x: torch.as_tensor(np.ascontiguousarray(x), device="cuda")
    with torch.no_grad():
        if kind == "frames":
            h, b = _dam_break(case, seed)
            return _dense64(dev(h.astype(np.float32)).double(), dev(b), 1.0, case["bc"], 0.0, 0.0, False,
                            t_end=case["frame_s"])
        if kind == "dense":
            if case["nx"] * case["ny"] > 4.0e7:       # the float64 fields would not be quick
                return None
            b = _slope_bed(case, seed).double()
            q = _dense64(torch.full_like(b, SLOPE_H0), b, SLOPE_DX, "fall", SLOPE_N, SLOPE_RAIN, True,
                         steps=SLOPE_WARM + case["steps"])
            return [q[0], q[1], q[2]]
        if kind == "coastal":
            if case["tail"]:
                return None
            c = _Coast64(_coast_fields(case["n"], seed, case["dtype"]), case["dtype"])
            q, top = c.run(COAST_WARM + case["steps"])
            k = NGH
            if case["layout"] == "dense":
                # the dense form also carries the cells outside the active set, through a step with
                # no fluxes; they rest in these cases
                out = [x[k:-k, k:-k] for x in q]
                # its running maximum starts from the first step on every cell
                return out + ([_sel(c.act, top, c.q[0])[k:-k, k:-k]] if case["maxh"] else [])
            return [x[c.stored] for x in q] + ([top[c.stored]] if case["maxh"] else [])
        if kind == "ensemble":
            out = []
            for m, n in enumerate(_sides(case)):
                c = _Coast64(_coast_fields(n, seed + 31 * m, "float32"), "float32")
                q, _ = c.run(COAST_WARM + case["steps"])
                out += [x[c.stored] for x in q]
            return out
    return _gradient64(case, seed)


def _gradient64(case: dict, seed: int):
    """The misfit and its gradient by autograd through the float64 steps, one step at a time."""
    if case["n"] ** 2 * case["steps"] > 1.2e8:       # autograd would not be quick
        return None
    from torch.utils.checkpoint import checkpoint
    c = _Coast64(_coast_fields(case["n"], seed, "float32"), "float32")
    ids = _gauge_ids(c.act[c.stored].cpu().numpy(), c.q[0][c.stored].float().cpu().numpy(), seed)
    with torch.no_grad():                             # the time steps, frozen
        q, t, dts = c.q, 0.0, []
        for _ in range(case["steps"]):
            dts.append(_dt64(q, c.act, COAST_DX))
            q = c.step(q, c.b, c.ntab, t, dts[-1])
            t += dts[-1]
    flat = torch.nonzero(c.stored.reshape(-1))[:, 0]
    at = flat[torch.as_tensor(ids, device="cuda")]

    def depths(ntab, b, keep):
        q, t, got = c.q, 0.0, []
        for dt in dts:
            if keep:
                q = checkpoint(lambda x, y, z, t=t, dt=dt: c.step(x, y, z, t, dt), q, b, ntab, use_reentrant=False)
            else:
                q = c.step(q, b, ntab, t, dt)
            t += dt
            got.append(q[0].reshape(-1)[at])
        return torch.stack(got)

    with torch.no_grad():
        seen = depths((c.ntab * torch.as_tensor(_truth(seed), device="cuda")).float().double(), c.b, False)
    ntab = c.ntab.clone().requires_grad_(True)
    bed = c.b.reshape(-1)[flat].clone().requires_grad_(True)
    b = c.b.reshape(-1).index_put((flat,), bed).reshape(c.b.shape)
    loss = ((depths(ntab, b, True) - seen) ** 2).sum()
    loss.backward()
    return {"loss": loss.detach(), "n": ntab.grad, "bed": bed.grad}
