"""Launches of the general path with up to 12 ring cells, on grids that one
round of workgroups covers: a call of n steps, which takes the deepest launches
there, against n calls of one step, bit for bit (a cell's arithmetic does not
depend on its tile or on where launches split)."""
import numpy as np
import pytest

import yolohtli_amd as Y
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu

ANISO = dict(anisotropy=1, diff_par=0.0016, diff_per=0.0006, degrad=30.0)
RULES = [  # (mask, options, a call's steps: one launch of the deepest, and a remainder)
    (0, dict(timeIntOrder=4), (3, 7)),
    (0, dict(timeIntOrder=2, **ANISO), (3, 5)),
    (1, dict(timeIntOrder=2), (5, 6, 13)),
    (0, dict(neumannBC=0, boundaryVal=0.1), (11, 12, 17)),
    (0, dict(lap4=1), (9, 12, 25)),
]


@pytest.mark.parametrize("rule", range(len(RULES)))
@pytest.mark.parametrize("nx,ny", [(4, 4), (40, 24), (41, 25), (128, 128), (201, 699)])
def test_deep_launches_equal_single_steps(torch_cuda, nx, ny, rule):
    masked, over, calls = RULES[rule]
    rng = np.random.default_rng(nx + rule)
    p = T.grid_params(nx, ny, solidSwitch=masked, **over)
    m = (rng.random(nx * ny) > 0.1).astype(np.uint8) if masked else np.ones(nx * ny, np.uint8)
    f = [rng.random(nx * ny).astype(np.float32) * m for _ in range(2)]
    plans = [Y.Plan(p) for _ in range(2)]
    for pl in plans:
        if masked:
            pl.set_mask(m)
        pl.set_state(*f)
    for n in calls:
        plans[0].step(n)
        for _ in range(n):
            plans[1].step(1)
        for a, b in zip(plans[0].get_state(), plans[1].get_state()):
            np.testing.assert_array_equal(a, b)
    for pl in plans:
        pl.close()
