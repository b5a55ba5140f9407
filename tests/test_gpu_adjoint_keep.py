"""The gradient with every state kept (up to 4 GiB of them) against the one
with checkpoints and recomputed segments.

1024 x 1024 states take 12.58 MB each: 341 of them (340 steps) are kept, 346
(345 steps) are not.  Only step 340 is recorded, so both runs have the same
loss and gradient; the steps after it carry lambda = 0.  Forward and lambda
agree bit for bit; the FP64 sums of the gradients group the same terms
differently: 1e-12.
"""
import numpy as np
import pytest

from yolohtli_amd.adjoint import SensorProblem, adjoint_workload

pytestmark = pytest.mark.gpu


def test_kept_states_equal_recomputed_segments(torch_cuda):
    torch = torch_cuda
    n = 1024
    p, x0, _, D_hidden, _ = adjoint_workload(n=n, nsteps=345, nsensors=8, config=43)
    rng = np.random.default_rng(9)
    sensors = np.sort(rng.choice(n, 32, replace=False) * n + rng.integers(40, 80, 32))
    D = torch.from_numpy(D_hidden.reshape(-1)).cuda()
    out = []
    for nsteps in (340, 345):
        pr = SensorProblem(p, nsteps, sensors, x0, rec_every=340, ckpt_every=90)
        pr.set_targets(np.full((1, 32), 0.3, np.float32))
        L, tr = pr.forward(D)
        gD, gt = pr.backward()
        out.append((L, tr, gD.cpu().numpy(), gt))
        pr.close()
    assert out[0][0] == out[1][0] and out[0][0] > 0
    np.testing.assert_array_equal(out[0][1], out[1][1])
    scale = np.abs(out[0][2]).max()
    assert scale > 0
    np.testing.assert_allclose(out[1][2], out[0][2], rtol=1e-12, atol=1e-12 * scale)
    np.testing.assert_allclose(out[1][3], out[0][3], rtol=1e-12)
