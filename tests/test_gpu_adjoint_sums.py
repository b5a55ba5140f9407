"""dL/dD of one step, cell by cell: products and sums over a cell's links in FP64.

After one recorded step lambda is the sensors' source alone, so dL/dD of a
sensor's cell is mu times the sum of r (u_n - u) over its links and of a
neighbour's cell r L (u - u_n), with r, mu, L and the differences of u in FP32 as
the library has them.  The sums of four random terms differ from that by FP64
rounding, 4 * 1.1e-16 of the terms; sums in FP32 by 1e-8.
"""
import numpy as np
import pytest

import yolohtli_amd as Y
from yolohtli_amd import abi_types as T
from yolohtli_amd.adjoint import SensorProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 8])
def test_link_sums_in_fp64(torch_cuda, k):
    torch = torch_cuda
    nx, ny = 57, 43
    p = T.grid_params(nx, ny, model=T.YH_MODEL_3V_FK, heaviside_width=0.01)
    p.Ly = 0.035 * (ny - 1)
    rng = np.random.default_rng(12)
    x0 = [rng.random(nx * ny).astype(np.float32) for _ in range(3)]
    sensors = np.array([i + nx * j for j in range(2, ny - 2, 4) for i in range(2, nx - 2, 4)], np.int32)
    targets = np.full((1, len(sensors)), 0.3, np.float32)
    pr = SensorProblem(p, 1, sensors, x0)
    pr.set_substeps(k)
    pr.set_targets(targets)
    _, tr = pr.forward(torch.full((nx * ny,), 0.001, device="cuda"))
    gD = pr.backward()[0].cpu().numpy().reshape(ny, nx)
    pr.close()
    lam = np.zeros(nx * ny, np.float32)
    lam[sensors] = (2.0 * (tr[0].astype(np.float64) - targets[0])).astype(np.float32)
    lam = lam.reshape(ny, nx)
    d = Y.derive(p)
    r = [np.float32(0.5 * p.tc * d.dt / h ** 2) for h in (d.hx, d.hx, d.hy, d.hy)]
    u = x0[0].reshape(ny, nx)
    want, scale = np.zeros((ny, nx)), 0.0
    for q, (dy, dx) in enumerate(((0, -1), (0, 1), (1, 0), (-1, 0))):
        un, ln = np.roll(u, (-dy, -dx), (0, 1)), np.roll(lam, (-dy, -dx), (0, 1))
        term = float(r[q]) * (lam - ln).astype(np.float64) * (un - u).astype(np.float64)
        want[1:-1, 1:-1] += term[1:-1, 1:-1]
        scale = max(scale, np.abs(term).max())
    assert scale > 0
    assert np.abs(gD - want).max() < 1e-14 * scale
