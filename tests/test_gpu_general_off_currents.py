"""Fenton-Karma steps of the general path with a time constant that switches its
current or gate off: infinite, past the range of a float, or (tau_si, which is
doubled) just below it.  Oracle: the same steps with 1e30, which in 64 bits moves
no value by more than 1e-28.  Tolerance as in test_gpu_general.py.
"""
import numpy as np
import pytest

import oracle.oracle as O
import yolohtli_amd as Y
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu

TAUS = ("tau_d", "tau_r", "tau_si", "tau_0", "tau_vp", "tau_v1m", "tau_v2m", "tau_wp", "tau_wm")


@pytest.mark.parametrize("tau,value", [(t, float("inf")) for t in TAUS] +
                         [("tau_0", 1e39), ("tau_si", 2e38)])
@pytest.mark.parametrize("over", [dict(timeIntOrder=4), dict(neumannBC=0)])
def test_off_currents(torch_cuda, tau, value, over):
    nx, ny = 70, 52
    p, q = (T.grid_params(nx, ny, model=T.YH_MODEL_3V_FK, fk={tau: v}, **over)
            for v in (value, 1e30))
    rng = np.random.default_rng(31)
    f = list(Y.initGates(nx, ny, u_cols=12, rest=1.0, refr=0.0, nvars=3))
    f[0] = np.clip(f[0] + 0.05 * rng.random(nx * ny).astype(np.float32), 0, 1)
    pl = Y.Plan(p)
    pl.set_state(*f)
    pl.step(40)
    got = pl.get_state()
    pl.close()
    want = O.run_general(q, [x.astype(np.float64) for x in f], 40)
    for a in range(3):
        assert np.isfinite(got[a]).all()
        assert np.mean(np.abs(got[a] - want[a]) > 1e-4) < 2e-3
