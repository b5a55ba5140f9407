"""The previous u of the general path's calls (the tip test's input): a launch of
several steps writes it, a single step leaves it in the other state buffer."""
import numpy as np
import pytest

import yolohtli_amd as Y
from timing import ratio
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


@pytest.mark.parametrize("over,stim", [(dict(), True), (dict(neumannBC=0), False),
                                       (dict(timeIntOrder=2), False)])
def test_first_call_under_capture(torch_cuda, over, stim):
    """The first call of a plan, recorded into a graph: nothing is allocated, and
    every replay takes the state to the same steps as an eager call; eager
    calls follow."""
    torch = torch_cuda
    nx, ny = 90, 70
    p = T.grid_params(nx, ny, **over)
    f = Y.initGates(nx, ny)
    cap, ref = Y.Plan(p), Y.Plan(p)
    side = torch.cuda.Stream()
    for pl in (cap, ref):
        pl.set_state(*f)
        if stim:
            pl.set_stimulus(True, (30, 20))
    ref.step(4)
    want = ref.get_state()
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=side):
        cap.step(4)
    buf = [x.copy() for x in f]
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        buf = cap.get_state()
    # four steps in an odd number of launches leave the state they started from
    # alone, in an even number they go on from their own result
    for _ in range(2):
        if all(np.array_equal(x, y) for x, y in zip(buf, want)):
            break
        ref.step(4)
        want = ref.get_state()
    for x, y in zip(buf, want):
        np.testing.assert_array_equal(x, y)
    for pl in (cap, ref):
        pl.step(5)
        pl.track_tips()
    for x, y in zip(cap.get_state(), ref.get_state()):
        np.testing.assert_array_equal(x, y)
    for pl in (cap, ref):
        pl.close()


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
    least = ratio(torch, lambda: pl.step(1), lambda: Y.reactionDiffusion_wrapper(p, b, a), 20, 1.1)
    pl.close()
    assert least < 1.1
