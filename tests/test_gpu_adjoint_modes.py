"""The gradient with checkpoints (keep_bytes=0) against the one with every state
kept: masked and not, one-step and tiled launches, checkpoints closer together than
a launch is deep and not, records inside earlier segments, a ragged grid.

Forward and lambda agree bit for bit; the FP64 sums group the same terms
differently: 1e-12.  That the kept one is right is test_gpu_adjoint_axes.py's.
"""
import numpy as np
import pytest

from yolohtli_amd import abi_types as T
from yolohtli_amd.adjoint import SensorProblem, adjoint_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("k", [1, 8])
@pytest.mark.parametrize("ckpt", [3, 70, 240])
def test_checkpoints_equal_kept_states(torch_cuda, masked, k, ckpt):
    torch = torch_cuda
    nx, ny, nsteps = 53, 35, 240
    base = adjoint_workload(n=64, nsteps=nsteps, nsensors=8, config=44)[0]
    p = T.copy_params(base, nx=nx, ny=ny, Lx=0.025 * (nx - 1), Ly=0.035 * (ny - 1),
                      solidSwitch=int(masked))
    rng = np.random.default_rng(3)
    solid = (rng.random(nx * ny) > 0.03).astype(np.uint8) if masked else None
    j, i = np.divmod(np.arange(nx * ny), nx)
    x0 = [np.where(i < 5, 1.0, 0.0) * np.where(j < ny // 2 + 1, 1.0, 0.2),
          np.full(nx * ny, 0.9), np.full(nx * ny, 0.8)]
    D = torch.from_numpy((0.001 * (1 + 0.2 * rng.random(nx * ny))).astype(np.float32)).cuda()
    sensors = np.sort(rng.choice(np.flatnonzero(i < 16), 8, replace=False)).astype(np.int32)
    out = []
    for keep in (None, 0):
        pr = SensorProblem(p, nsteps, sensors, x0, rec_every=4, ckpt_every=ckpt, mask=solid,
                           keep_bytes=keep)
        assert pr.keeps_states == (keep is None)
        pr.set_substeps(k)
        pr.set_targets(np.full((nsteps // 4, 8), 0.3, np.float32))
        L, tr = pr.forward(D)
        gD, gt = pr.backward()
        out.append((L, tr, gD.cpu().numpy(), gt))
        pr.close()
    assert out[0][0] == out[1][0] > 0
    np.testing.assert_array_equal(out[0][1], out[1][1])
    for q in (2, 3):
        scale = np.abs(out[0][q]).max()
        assert scale > 0
        np.testing.assert_allclose(out[1][q], out[0][q], rtol=1e-12, atol=1e-12 * scale)


def test_the_limit(torch_cuda):
    """1024 x 1024 states take 12.58 MB each; the default keeps up to 4 GiB."""
    p, x0, sensors, _, _ = adjoint_workload(n=1024, nsteps=10, nsensors=8)
    for nsteps, keep, kept in ((340, None, True), (341, None, False), (10, 11 * 3 << 22, True),
                               (10, (11 * 3 << 22) - 1, False), (1, 0, False)):
        pr = SensorProblem(p, nsteps, sensors, x0, keep_bytes=keep)
        assert pr.keeps_states == kept
        pr.close()
