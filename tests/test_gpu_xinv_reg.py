"""The inverse x kernel with the lines in registers (nxp/2 = 2^a 3^b from 16 to
256; z splits 1, 2, 3, 4, 6, 8, 9): each line length with each split, tiles of one
column, of a column count that is no power of two and partial ones, a single
y row, the duplicate row of a periodic y, z walls, P with its ghosts.

FP64: the parity bar against the C oracle.  FP32+refine: one sweep leaves the
square of the FP32 solve's error (below 1e-5 on these grids), 1e-10.  A batch
runs the same arithmetic as the plans one by one: equal bits."""
from __future__ import annotations

import pytest

import dfp
from _cases import fields, make_grid, oracle_project, rel_linf

pytestmark = pytest.mark.gpu

DT, C3 = 1e-3, 0.75


def _check(g, tuning=None, precision=dfp.DFP_FP64, bar=1e-12):
    U, V, W, P, rhs = fields(g, 3, 0.1)
    o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    oracle_project(g, *o, DT, C3, save_p=True)
    plan = dfp.Plan(g, precision=precision, tuning=tuning)
    plan.project(U, V, W, rhs, P, DT, C3, save_p=True)
    plan.close()
    for lab, a, b in zip(("U", "V", "W", "P", "phi"), (U, V, W, P, rhs), o):
        assert rel_linf(a, b) <= bar, lab


@pytest.mark.parametrize("nxp", [32, 48, 54, 64, 72, 96, 108, 128, 144, 162, 192, 216, 256, 288, 324, 384, 432, 512])
@pytest.mark.parametrize("nym,nzp,R,T", [(1, 16, 1, 0), (3, 16, 2, 0), (9, 16, 4, 0), (4, 24, 8, 0), (6, 12, 4, 3),
                                         (5, 16, 4, 1), (7, 6, 1, 2),
                                         (4, 12, 3, 0), (3, 24, 6, 0), (5, 27, 9, 0)])
def test_lines_in_registers_match_oracle(nxp, nym, nzp, R, T):
    if R * T * (nxp // 2) > 2048:
        pytest.skip("a plan takes no tile of that many points")
    print(f"{nxp}x{nym}x{nzp}, split {R}, columns {T}", flush=True)
    g = make_grid(nxp, nym, nzp, 1.5)
    _check(g, (R, T, 0, 0))
    _check(g, (R, T, 0, 0), dfp.DFP_FP32_REFINE, 1e-10)


@pytest.mark.parametrize("nxp", [32, 54, 96, 108, 128, 162, 512])
def test_lines_in_registers_periodic_y_and_z_walls(nxp):
    print(f"nxp {nxp}", flush=True)
    _check(dfp.periodic_y_grid(nxp, 9, 16))
    _check(dfp.duct_grid(nxp, 6, 10, 1.0, 0.7))


@pytest.mark.parametrize("precision", [dfp.DFP_FP64, dfp.DFP_FP32_REFINE])
def test_batch_of_register_lines_equals_single_plans(precision):
    import torch

    from dfp.batch import Batch, Case

    sizes = [(32, 5, 12), (64, 7, 16), (128, 4, 24), (256, 3, 16), (512, 2, 16), (48, 6, 12), (96, 5, 24), (36, 4, 12), (54, 3, 16),
             (162, 4, 16), (324, 2, 12), (432, 2, 12)]
    batch, cases, singles = Batch(max_cases=len(sizes)), [], []
    for n in sizes:
        g = make_grid(*n, 1.5)
        host = fields(g, sum(n), 0.1)
        dev = [[torch.from_numpy(a.T.copy()).cuda() for a in host] for _ in range(2)]
        U, V, W, P, rhs = dev[0]
        plan = dfp.Plan(g, precision=precision)
        plan.project(U, V, W, rhs, P, DT, C3, save_p=True)
        plan.close()
        singles.append(dev[0])
        U, V, W, P, rhs = dev[1]
        cases.append(Case(dfp.Plan(g, precision=precision), U, V, W, rhs, P, DT, C3, save_p=True))
    batch.project(cases)
    for n, c, s in zip(sizes, cases, singles):
        for lab, a, b in zip(("U", "V", "W", "P", "phi"), (c.U, c.V, c.W, c.P, c.rhs), s):
            assert torch.equal(a, b), (n, lab)


@pytest.mark.parametrize("nxp", [32, 54, 72, 108, 128, 162, 192, 324, 512])
@pytest.mark.parametrize("nym,nzp,R,T", [(3, 16, 2, 0), (9, 16, 4, 0), (1, 16, 1, 0), (4, 24, 8, 0), (5, 27, 9, 0)])
def test_solve_lines_in_registers_match_oracle(nxp, nym, nzp, R, T):
    """The right-hand side's forward transform in registers: phi of a solve, alone and in a batch (equal bits)."""
    import numpy as np
    import torch

    from dfp.batch import Batch, Case

    print(f"solve {nxp}x{nym}x{nzp}, split {R}", flush=True)
    g = make_grid(nxp, nym, nzp, 1.5)
    U, V, W, P, rhs = fields(g, 5, 0.1)
    o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    oracle_project(g, *o, DT, C3, save_p=False)
    plan = dfp.Plan(g, tuning=(R, T, 0, 0))
    plan.divergence(U, V, W, rhs)
    b = rhs.copy(order="F")
    plan.solve(rhs)
    assert rel_linf(rhs, o[4]) <= 1e-12
    dev = torch.from_numpy(b.T.copy()).cuda()
    Batch(max_cases=1).project([Case(plan, None, None, None, dev)], solve_only=True)
    assert np.array_equal(dev.cpu().numpy().T, rhs)
    plan.close()
