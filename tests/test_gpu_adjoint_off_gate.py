"""Loss and gradient with v's recovery above u_v switched off (tau_v2- infinite, or
past the range of a float) against the FP64 oracle with 1e30 (with 1e26 it gives
the same bits).  Tolerance as in test_gpu_adjoint_axes.py.
"""
import numpy as np
import pytest

import oracle.oracle as O
from yolohtli_amd import abi_types as T
from yolohtli_amd.adjoint import SensorProblem, adjoint_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 8])
@pytest.mark.parametrize("value", [float("inf"), 1e39])
def test_gradient_without_recovery(torch_cuda, value, k):
    torch = torch_cuda
    n, nsteps = 40, 160
    base = adjoint_workload(n=n, nsteps=nsteps, nsensors=8, config=45)[0]
    p, q = (T.copy_params(base, fk={"tau_v2m": v}) for v in (value, 1e30))
    rng = np.random.default_rng(4)
    j, i = np.divmod(np.arange(n * n), n)
    u = np.where(i < 5, 1.0, 0.0) * np.where(j < n // 2, 1.0, 0.2)
    x0 = [u.astype(np.float32), np.full(n * n, 0.9, np.float32), np.full(n * n, 0.8, np.float32)]
    D = (0.001 * (1 + 0.2 * rng.random(n * n))).astype(np.float32)
    sensors = np.sort(rng.choice(np.flatnonzero(i < 14), 8, replace=False)).astype(np.int32)
    targets = np.full((nsteps // 4, 8), 0.3, np.float32)
    pr = SensorProblem(p, nsteps, sensors, x0, rec_every=4)
    pr.set_substeps(k)
    pr.set_targets(targets)
    L, _ = pr.forward(torch.from_numpy(D).cuda())
    gD, gt = pr.backward()
    pr.close()
    Lo, gDo, gto = O.fk_adjoint(q, D.astype(np.float64), [x.astype(np.float64) for x in x0], nsteps,
                                4, sensors, targets.astype(np.float64), None)
    assert L == pytest.approx(Lo, rel=1e-4)
    assert np.linalg.norm(gD.cpu().numpy() - gDo) < 1e-4 * np.linalg.norm(gDo)
    np.testing.assert_allclose(gt, gto, rtol=1e-4, atol=1e-4 * np.abs(gto).max())
