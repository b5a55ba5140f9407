"""The host's share of a yh_step_noalloc call: one step, calls back to back, is one
launch, as yh_rd_step_dev is (1.4 leaves room for the argument checks and the clock;
with the launch table made on every call it took twice as long).  Calls of
alternating grids and models keep their tables; a call of more grids than are kept
gives the same bits."""
import ctypes as C

import numpy as np
import pytest

import yolohtli_amd as Y
from timing import ratio
from yolohtli_amd import abi_types as T
from yolohtli_amd._lib import lib

pytestmark = pytest.mark.gpu


def _arrays(torch, p):
    nv = T.nvars(p)
    f = Y.init_random(p.nx, p.ny, 5, nvars=nv)
    a = [torch.from_numpy(x).cuda() for x in f]
    b = [torch.empty_like(x) for x in a]
    ptrs = [(C.c_void_p * 3)(*[x.data_ptr() for x in t]) for t in (b, a)]
    return a, b, ptrs, f


@pytest.mark.parametrize("model", [T.YH_MODEL_2V_REF, T.YH_MODEL_3V_FK])
def test_one_step_is_one_launch(torch_cuda, model):
    torch = torch_cuda
    sets = [(p, *_arrays(torch, p)) for p in (T.grid_params(n, n, model=model) for n in (64, 200, 256))]
    s = torch.cuda.current_stream().cuda_stream

    def calls(fn):
        for p, _, _, (o, i), _ in sets:
            assert fn(p, o, i) == 0

    assert ratio(torch,
                 lambda: calls(lambda p, o, i: lib().yh_step_noalloc(C.byref(p), o, i, None, 1, s)),
                 lambda: calls(lambda p, o, i: lib().yh_rd_step_dev(C.byref(p), o, i, None, None, s)),
                 40, 1.4) < 1.4


def test_more_grids_than_are_kept(torch_cuda):
    torch = torch_cuda
    for _ in range(2):
        for n in range(40, 52):
            p = T.grid_params(n, n + 7, model=n % 2, diff_per=0.001 if n % 3 else 0.0006)
            a, b, (o, i), f = _arrays(torch, p)
            assert lib().yh_step_noalloc(C.byref(p), o, i, None, 17, None) == 0
            pl = Y.Plan(p)
            pl.set_state(*f)
            torch.cuda.synchronize()
            pl.step(17)
            for x, y in zip(b, pl.get_state()):
                np.testing.assert_array_equal(x.cpu().numpy(), y)
            pl.close()
