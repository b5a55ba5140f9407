"""The previous u of the general path's calls (the tip test's input): a launch of
several steps writes it, a single step leaves it in the other state buffer."""
import time

import numpy as np
import pytest

import yolohtli_amd as Y
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,masked", [(1, 1), (2, 0), (4, 0)])
def test_tips_do_not_depend_on_the_calls(torch_cuda, order, masked):
    """Random u, whose isolines u = Uth of two states cross in many cells."""
    nx, ny = 150, 131
    rng = np.random.default_rng(order)
    p = T.grid_params(nx, ny, timeIntOrder=order, solidSwitch=masked,
                      neumannBC=0 if order == 1 else 1, Uth=0.5)
    f = [rng.random(nx * ny).astype(np.float32) for _ in range(2)]
    logs = []
    for calls in ((5, 1, 7), (1,) * 13, (12, 1), (3, 2, 1, 7)):
        pl = Y.Plan(p)
        if masked:
            pl.set_mask(Y.make_holes(nx, ny, 6, 2.0, 6.0, 3))
        pl.set_state(*f)
        done = 0
        for n in calls:
            pl.step(n)
            done += n
            if done in (6, 13):
                pl.track_tips()
        if 6 in np.cumsum(calls):
            logs.append(pl.read_tips())
        pl.close()
    assert len(logs) == 3 and len(logs[0]) > 0
    for log in logs[1:]:
        np.testing.assert_array_equal(log, logs[0])


def test_single_step_moves_no_more_than_the_wrapper(torch_cuda):
    """One Dirichlet step of a plan and of the wrapper on a grid bound by
    memory: the plan has no other field to write (10% are for the clock)."""
    torch = torch_cuda
    n = 4096
    p = T.grid_params(n, n, neumannBC=0)
    f = Y.initGates(n, n)
    pl = Y.Plan(p)
    pl.set_state(*f)
    a = [torch.from_numpy(x).cuda() for x in f]
    b = [torch.empty_like(x) for x in a]
    best = [float("inf")] * 2
    for _ in range(8):
        for q, one in enumerate((lambda: pl.step(1),
                                 lambda: Y.reactionDiffusion_wrapper(p, b, a))):
            one()
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                one()
            torch.cuda.synchronize()
            best[q] = min(best[q], time.perf_counter() - t)
    pl.close()
    assert best[0] < 1.1 * best[1]
