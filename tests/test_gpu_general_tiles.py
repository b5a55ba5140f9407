"""Edges of the tiles of the general path (general.hip k_general): grids from
the smallest accepted size over one region to ragged multiples of the output
tile, each neighbour rule, step counts that leave remainders of the fused
steps.

Tolerance: one FP32 step of these branches is within 3e-6 of the FP64 oracle
(tests/test_gpu_general.py), so 5 steps of the smooth 2V model within 1.5e-5.
A cell's arithmetic does not depend on its tile or on where launches split, so
one call of n steps equals n calls of one step bit for bit.
"""
import numpy as np
import pytest

import oracle.oracle as O
import yolohtli_amd as Y
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu

ANISO = dict(anisotropy=1, diff_par=0.0016, diff_per=0.0006, degrad=30.0)
RULES = [
    (0, dict(timeIntOrder=4, lap4=1)),
    (0, dict(timeIntOrder=2, **ANISO)),
    (0, dict(timeIntOrder=4, lap4=1, **ANISO)),
    (0, dict(timeIntOrder=2, gateDiff=0)),
    (1, dict(timeIntOrder=2)),
    (1, dict(neumannBC=0, boundaryVal=0.1, **ANISO)),
]
SIZES = [(4, 4), (5, 67), (48, 32), (49, 33), (63, 9), (65, 130), (161, 47)]


def _plan(model, masked, over, nx, ny, seed):
    rng = np.random.default_rng(seed)
    p = T.grid_params(nx, ny, model=model, solidSwitch=masked, **over)
    f = [rng.random(nx * ny).astype(np.float32) for _ in range(T.nvars(p))]
    m = (rng.random(nx * ny) > 0.15).astype(np.uint8) if masked else None
    if masked:
        f = [x * m for x in f]
    pl = Y.Plan(p)
    if masked:
        pl.set_mask(m)
    pl.set_state(*f)
    return p, pl, f, m


@pytest.mark.parametrize("rule", range(len(RULES)))
@pytest.mark.parametrize("nx,ny", SIZES)
def test_tile_edges_match_oracle(torch_cuda, nx, ny, rule):
    masked, over = RULES[rule]
    p, pl, f, m = _plan(T.YH_MODEL_2V_REF, masked, over, nx, ny, 900 + rule)
    pl.step(5)
    got = pl.get_state()
    pl.close()
    want = O.run_general(p, [x.astype(np.float64) for x in f], 5, solid=m)
    for g, w in zip(got, want):
        assert np.abs(g - w.reshape(-1)).max() < 1.5e-5


@pytest.mark.parametrize("model", [T.YH_MODEL_2V_REF, T.YH_MODEL_3V_FK])
@pytest.mark.parametrize("rule", range(len(RULES)))
def test_one_call_equals_single_steps(torch_cuda, model, rule):
    """State, the previous u the tip test reads, and the APD state."""
    masked, over = RULES[rule]
    out = []
    for calls in ([9], [1] * 9, [2, 3, 4]):
        p, pl, f, m = _plan(model, masked, over, 113, 75, 950 + rule)
        pl.apd_enable(0.4)
        for n in calls:
            pl.step(n)
        pl.track_tips()
        out.append((pl.get_state(), pl.read_tips(), pl.apd_get()))
        pl.close()
    for state, tips, apd in out[1:]:
        for a, b in zip(state, out[0][0]):
            np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(tips, out[0][1])
        for k in apd:
            np.testing.assert_array_equal(apd[k], out[0][2][k])
