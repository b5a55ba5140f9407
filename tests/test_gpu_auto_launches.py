"""The launches of a plan left on AUTO (plan.cpp auto_table: mixed tile shapes
and depths) against launches of one step each of one fixed shape: a cell's
value depends on neither, so state, tips and step counts agree bit for bit.
Grids from the smallest accepted to several rounds of workgroups, step counts
below, at and above the table's end (48) and with odd remainders.
"""
import numpy as np
import pytest

import yolohtli_amd as Y
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu

SIZES = [(4, 4), (5, 41), (17, 33), (100, 37), (333, 129), (800, 800), (1301, 702)]
STEPS = [1, 2, 7, 20, 48, 49, 61, 115]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("model,masked,ratio", [(0, 0, 1.0), (0, 1, 0.4), (1, 0, 0.4), (1, 1, 1.0)])
def test_auto_equals_single_steps(torch_cuda, nx, ny, model, masked, ratio):
    rng = np.random.default_rng(nx + 7 * ny + model)
    p = T.grid_params(nx, ny, model=model, solidSwitch=masked, diff_per=0.001 * ratio)
    f = [rng.random(nx * ny).astype(np.float32) for _ in range(2 + model)]
    m = (rng.random(nx * ny) > 0.05).astype(np.uint8)
    out = []
    for auto in (True, False):
        pl = Y.Plan(p)
        if masked:
            pl.set_mask(m)
        pl.set_state(*f)
        if not auto:
            pl.set_kernel(T.YH_KERNEL_TILED, 1, 4, 8, 1)
        for n in STEPS:
            pl.step(n)
            pl.track_tips()
        out.append((pl.get_state(), pl.read_tips(), pl.step_count()))
        pl.close()
    for a, b in zip(out[0][0], out[1][0]):
        np.testing.assert_array_equal(a, b)
    np.testing.assert_array_equal(out[0][1], out[1][1])
    assert out[0][2] == out[1][2] == sum(STEPS)
