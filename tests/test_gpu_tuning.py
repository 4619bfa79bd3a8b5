"""Launch shapes: those that a plan reports make the same plan again, and x
columns do not change FP64 results."""
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


@pytest.mark.parametrize("grid", [dfp.periodic_y_grid(32, 33, 32), dfp.periodic_y_grid(32, 25, 18),
                                  dfp.duct_grid(32, 12, 20, 1.2, 0.8), dfp.zwall_periodic_y_grid(32, 13, 20, 0.8),
                                  dfp.channel_grid(32, 12, 24, 1.2, x_bc_type=1)],
                         ids=["planes", "lds", "duct", "zwall", "inflow"])
def test_reported_shapes_of_every_branch_make_the_same_plan(grid):
    print(f"{grid.nxp}x{grid.nym}x{grid.nzp}", flush=True)
    host = fields(grid, 3, 0.1)
    plan = dfp.Plan(grid)
    again = dfp.Plan(grid, tuning=plan.tuning)
    assert again.tuning == plan.tuning
    for a, b in zip(_project(plan, host), _project(again, host)):
        assert np.array_equal(a, b)
    plan.close()
    again.close()


@pytest.mark.parametrize("precision", [dfp.DFP_FP64, dfp.DFP_FP32_REFINE], ids=["fp64", "fp32"])
def test_reported_lds_shape_makes_the_same_plan(precision):
    g = make_grid(32, 20, 64, 1.5)
    plan = dfp.Plan(g, precision=precision, tuning=(4, 0, 0, 2))
    again = dfp.Plan(g, precision=precision, tuning=plan.tuning)
    assert again.tuning == plan.tuning and plan.tuning[3] == 2
    host = fields(g, 3, 0.1)
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


@pytest.mark.parametrize("size,split,columns", [((128, 5, 64), 4, (1, 4, 8, 16)), ((128, 5, 16), 1, (2, 16)),
                                                ((32, 3, 256), 4, (1, 32, 64)), ((96, 4, 64), 4, (1, 8, 16)),
                                                ((162, 6, 36), 4, (1, 3, 9)), ((54, 7, 108), 4, (3, 9, 27)),
                                                ((512, 2, 16), 4, (1, 2, 4)), ((64, 40, 64), 4, (1, 2, 16))])
def test_columns_do_not_change_fp64_results(size, split, columns):
    """Tiles below and above what the register x kernels hold (2048 points): the same kernels, the same bits."""
    print(f"{size} split {split} columns {columns}", flush=True)
    g = make_grid(*size, 1.5)
    host = fields(g, 5, 0.1)
    ref = None
    for T in columns:
        plan = dfp.Plan(g, tuning=(split, T, 0, 0))
        assert plan.tuning[1] == T
        out = list(_project(plan, host))
        rhs = host[4].copy(order="F")
        plan.divergence(*(a.copy(order="F") for a in host[:3]), rhs)
        plan.solve(rhs)
        out.append(rhs)
        plan.close()
        for a, b in zip(out, ref or out):
            assert np.array_equal(a, b), T
        ref = ref or out


@pytest.mark.parametrize("T", [4, 16])
def test_batched_columns_equal_single_plans(T):
    from dfp.batch import Batch, Case

    g = make_grid(128, 5, 64, 1.5)
    host = fields(g, 6, 0.1)
    plan = dfp.Plan(g, tuning=(4, T, 0, 0))
    div = host[4].copy(order="F")
    plan.divergence(*(a.copy(order="F") for a in host[:3]), div)
    for solve_only in (False, True):
        one, two = ([dfp.DeviceArray.from_host(a) for a in (*host[:4], div)] for _ in range(2))
        U, V, W, P, rhs = one
        if solve_only:
            plan.solve(rhs, P, DT, C3, save_p=True)
        else:
            plan.project(U, V, W, rhs, P, DT, C3, save_p=True)
        U, V, W, P, rhs = two
        batch = Batch(max_cases=1)
        batch.project([Case(plan, U, V, W, rhs, P, DT, C3, True)], solve_only=solve_only)
        for a, b in zip(one, two):
            assert np.array_equal(a.download(), b.download())
        batch.close()
    plan.close()
