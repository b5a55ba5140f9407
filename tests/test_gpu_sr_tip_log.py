"""The tips of a symmetry-reduction step in the plan's log, with more of them
than the lanes of the wave that moves them."""
import numpy as np
import pytest
import torch

import yolohtli_amd as Y
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [3, 14])
def test_first_step_logs_the_tips_of_its_rd_step(torch_cuda, waves):
    """A step at count 0 logs the tips between the RD step of the state and the
    state.  The same fields come from a plain step and the tip search, so the
    counts agree, and the positions to 1e-3 cells (noise of 6e-8, an ulp of u,
    on the oracle's stepped u moves its tips by 1e-4 to 3e-4).  The oracle finds
    32 tips at 3 waves per axis and 756 at 14."""
    n = 192
    j, i = np.mgrid[0:n, 0:n] * (2 * np.pi * waves / n)
    p = T.grid_params(n, n, reduceSym=1, tipOffsetX=40, tipOffsetY=40)
    u = (p.Uth + 0.2 * np.sin(i) * np.cos(j)).astype(np.float32)
    v = (2 + 4 * np.sin(0.5 * i + 1.0) * np.sin(0.5 * j)).astype(np.float32)
    a = Y.Plan(p)
    a.set_state(u, v)
    a.sr_begin((n / 2, n / 2))
    a.sr_step(1)
    got = a.read_tips()
    a.close()
    b = Y.Plan(p)
    b.set_state(u, v)
    b.step(1)
    now = torch.from_numpy(np.ascontiguousarray(b.get_state()[0])).cuda()
    b.close()
    tips = torch.zeros((4096, 5), device="cuda")
    keys = torch.zeros(4096, dtype=torch.int32, device="cuda")
    count = torch.zeros(1, dtype=torch.int32, device="cuda")
    Y.tip_wrapper(p, now, torch.from_numpy(u).cuda(), 0.0, tips, keys, count, 4096)
    c = int(count)
    want = tips[:c][torch.argsort(keys[:c])].cpu().numpy()
    assert len(got) == c
    assert c == {3: 32, 14: 756}[waves]
    assert np.abs(got[:, :2] - want[:, :2]).max() < 1e-3
