"""The gradient on grids with two spacings and a ragged last tile, against the
FP64 oracle: x and y have their own weights, and the mirror terms of all four
edges lie in the same few tiles.

Tolerance: 1e-4.  The FP32 sweeps of 240 steps are off the oracle by about
2e-6 of the gradient's norm at these sizes (5e-6 after 600 steps of 64 x 64).
"""
import numpy as np
import pytest

import oracle.oracle as O
from yolohtli_amd import abi_types as T
from yolohtli_amd.adjoint import SensorProblem, adjoint_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("nx,ny,k", [(53, 35, 8), (35, 53, 1), (17, 4, 8)])
def test_gradient_with_two_spacings(torch_cuda, nx, ny, k, masked):
    torch = torch_cuda
    base = adjoint_workload(n=64, nsteps=240, nsensors=8, config=44)[0]
    p = T.copy_params(base, nx=nx, ny=ny, Lx=0.025 * (nx - 1), Ly=0.035 * (ny - 1),
                      solidSwitch=int(masked))
    rng = np.random.default_rng(nx)
    solid = None
    if masked:
        solid = (rng.random(nx * ny) > 0.03).astype(np.uint8)
    j, i = np.divmod(np.arange(nx * ny), nx)
    u = np.where(i < 5, 1.0, 0.0) * np.where(j < ny // 2 + 1, 1.0, 0.2)
    x0 = [u.astype(np.float32), np.full(nx * ny, 0.9, np.float32), np.full(nx * ny, 0.8, np.float32)]
    if masked:
        x0 = [x * solid for x in x0]
    D = (0.001 * (1 + 0.2 * rng.random(nx * ny))).astype(np.float32)
    cells = np.flatnonzero(i < 16) if solid is None else np.flatnonzero((i < 16) & (solid > 0))
    sensors = np.sort(rng.choice(cells, 8, replace=False)).astype(np.int32)
    targets = np.full((60, 8), 0.3, np.float32)
    pr = SensorProblem(p, 240, sensors, x0, rec_every=4, ckpt_every=70, mask=solid)
    pr.set_substeps(k)
    pr.set_targets(targets)
    L, _ = pr.forward(torch.from_numpy(D).cuda())
    gD, gt = pr.backward()
    pr.close()
    Lo, gDo, gto = O.fk_adjoint(p, D.astype(np.float64), [x.astype(np.float64) for x in x0], 240, 4,
                                sensors, targets.astype(np.float64), solid)
    assert L == pytest.approx(Lo, rel=1e-4)
    assert np.linalg.norm(gD.cpu().numpy() - gDo) < 1e-4 * np.linalg.norm(gDo)
    np.testing.assert_allclose(gt, gto, rtol=1e-4, atol=1e-4 * np.abs(gto).max())
