"""The launch shapes that a plan reports make the same plan again."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from _cases import fields, make_grid

pytestmark = pytest.mark.gpu

DT, C3 = 1e-3, 0.75


def _project(plan, host):
    U, V, W, P, rhs = (a.copy(order="F") for a in host)
    plan.project(U, V, W, rhs, P, DT, C3, save_p=True)
    return U, V, W, P, rhs


@pytest.mark.parametrize("size", [(16, 16, 16), (64, 40, 64), (54, 9, 27), (256, 6, 64), (512, 4, 64), (64, 260, 128)])
@pytest.mark.parametrize("precision", [dfp.DFP_FP64, dfp.DFP_FP32_REFINE], ids=["fp64", "fp32"])
def test_reported_shapes_make_the_same_plan(size, precision):
    """The library's own columns (one choice per x kernel, narrower on small grids) are reported as its choice: given
    back as a number they would set both kernels, which at 512 points in FP32 is refused."""
    print(f"{size} {precision}", flush=True)
    g = make_grid(*size, 1.5)
    host = fields(g, 3, 0.1)
    plan = dfp.Plan(g, precision=precision)
    assert plan.tuning[1] == 0
    again = dfp.Plan(g, precision=precision, tuning=plan.tuning)
    assert again.tuning == plan.tuning
    for a, b in zip(_project(plan, host), _project(again, host)):
        assert np.array_equal(a, b)
    plan.close()
    again.close()


def test_chosen_columns_are_reported():
    g = make_grid(64, 40, 64, 1.5)
    for T in (1, 4, 16):
        plan = dfp.Plan(g, tuning=(4, T, 0, 0))
        assert plan.tuning[:2] == (4, T)
        plan.close()
