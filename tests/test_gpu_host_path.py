"""Host paths of the step loops: the launches between two looks at a running clock, the statuses of
an ensemble in one read, and the torch wrapper of the adjoint with its tensors on the device."""
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,left,batch,want", [(0.125, 1.0, 64, 11), (0.1, 100.0, 64, 64), (0.1, 0.0, 64, 2),
                                                (0.1, -1.0, 64, 1), (0.0, 1.0, 64, 64), (float("nan"), 1.0, 8, 8),
                                                (0.5, 0.5, 1, 1), (1e-300, 1e9, 64, 64)])
def test_launches_to_the_end_of_a_run(dt, left, batch, want):
    from geoswe_amd import _lib as L
    c = L.GsClock()
    c.t, c.t_end, c.dt = 5.0, 5.0 + left, dt
    assert L.run_batch(c, batch) == want


@pytest.mark.parametrize("batch", [1, 7, 64])
def test_run_takes_the_same_steps_in_any_batch(gpu, batch):
    from geoswe_amd import Config, Mesh2D, Solver2D
    rng = np.random.default_rng(5)
    nx, ny = 40, 70
    bed = rng.random((nx, ny)).astype(np.float32)
    q = np.stack([np.maximum(1.4 - bed, 0), np.zeros((nx, ny)), np.zeros((nx, ny))]).astype(np.float32)
    q[0, :10] += 2.0                       # a dam break: dt shrinks as the front runs
    out = []
    for b in (batch, 1000):
        s = Solver2D(Mesh2D(nx, ny, 1.0, 1.0), Config(bc_x="wall", bc_y="wall", dtype="float32"), q, bed)
        n = [s.run(t, batch=b) for t in (0.5, 1.7, 1.7000001)]
        out.append((n, s.t, s.q_interior.copy()))
    assert out[0][0] == out[1][0] and out[0][1] == out[1][1] and np.array_equal(out[0][2], out[1][2])


ADJOINT = """
import itertools, sys
import numpy as np
import torch
torch.zeros(1, device="cuda")          # before the library, so that both share one HIP runtime
sys.path[:0] = [%r, %r]
from adjoint_cases import flowing_problem
from geoswe_amd.adjoint import GaugeMisfitFn
for dtype, td in itertools.product(("float32", "float64"), (torch.float32, torch.float64)):
    prob = flowing_problem(n=24, S=7, K=3, dtype=dtype)
    n0, b0 = prob.params()

    def run(device, strided=False):
        b = torch.as_tensor(b0, device=device).to(td)
        if strided:
            b = torch.stack([b, b + 1.0], 1)[:, 0]
            assert not b.is_contiguous()
        b = b.detach().requires_grad_(True)
        n = torch.tensor(n0, device=device, requires_grad=True)
        J = GaugeMisfitFn.apply(n, b, prob)
        (3.0 * J).backward()
        return [x.detach().cpu().numpy() for x in (J, n.grad, b.grad)]

    ref = run("cpu")
    assert np.abs(ref[2]).max() > 0
    runs = [run("cuda"), run("cuda", strided=True)]
    with torch.cuda.stream(torch.cuda.Stream()):
        runs += [run("cuda"), run("cuda")]
    for got in runs:
        for x, y in zip(ref, got):
            assert x.dtype == y.dtype and np.array_equal(x, y)
    try:
        GaugeMisfitFn.apply(torch.tensor(n0, device="cuda"), torch.zeros(3, device="cuda"), prob)
    except ValueError:
        print("ok", dtype, td, flush=True)
"""


def test_adjoint_wrapper_on_device_tensors(gpu):
    """Loss and gradients are the same bits with the tensors on the host, on the device, strided, and
    from a stream that does not wait for the default one; repeatedly, from the kept workspace. (A
    process of its own: torch finds the GPU only if it is set up before the library.)"""
    pytest.importorskip("torch")
    root = Path(__file__).resolve().parents[1]
    r = subprocess.run([sys.executable, "-c", ADJOINT % (str(root), str(root / "tests"))], capture_output=True,
                       text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.count("ok") == 4, r.stdout + r.stderr[-3000:]
