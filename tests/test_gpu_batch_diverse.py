"""Batches of many different sizes in one call: every stage then has many
launches (x kernels by z split and group of line lengths, z kernels by row
length), and the call takes them all.  Each case equals its own plan's bits."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from dfp.batch import Batch, Case
from _cases import fields, make_grid

pytestmark = pytest.mark.gpu

DT, C3 = 1e-3, 0.75
LINES = (16, 24, 27, 32, 36, 48, 54, 64, 72, 81, 96, 108, 128, 144, 162, 192, 216, 256)
ROWS = (8, 12, 16, 18, 24, 27, 32, 64)


def _sizes(n):
    """n cases (nxp, nym, nzp, z split): no two of the same split and line length, row lengths and counts mixed."""
    out = []
    for i in range(n):
        R = (1, 2, 3, 4, 6, 8, 9)[i % 7]
        out.append((2 * LINES[i % 18], (2, 3, 5, 9)[i % 4], R * ROWS[i % 8], R))
    assert len({(s[0], s[3]) for s in out}) == n
    return out


def _cases(n, precision=dfp.DFP_FP64, sweeps=None, solve_only=False):
    """Cases of n sizes, their fields on the host before a call, and after the same call of a single plan."""
    cases, start, want = [], [], []
    for i, (nxp, nym, nzp, R) in enumerate(_sizes(n)):
        g = make_grid(nxp, nym, nzp, 1.5)
        U, V, W, P, rhs = fields(g, i + 1, 0.1)
        plan = dfp.Plan(g, precision=precision, sweeps=sweeps, tuning=(R, 0, 0, 0))
        if solve_only:
            plan.divergence(U, V, W, rhs)
        start.append([a.copy(order="F") for a in (U, V, W, P, rhs)])
        if solve_only:
            plan.solve(rhs, P, DT, C3, save_p=True)
        else:
            plan.project(U, V, W, rhs, P, DT, C3, save_p=True)
        want.append((U, V, W, P, rhs))
        dev = [dfp.DeviceArray.from_host(a) for a in start[-1]]
        cases.append(Case(plan, *dev[:3], dev[4], dev[3], DT, C3, True))
    return cases, start, want


def _run(batch, part, cases, start, want, solve_only=False):
    for i in part:
        c = cases[i]
        for to, at in zip((c.U, c.V, c.W, c.P, c.rhs), start[i]):
            to.upload(at)
    batch.project([cases[i] for i in part], solve_only=solve_only)
    for i in part:
        c = cases[i]
        for lab, a, b in zip(("U", "V", "W", "P", "phi"), (c.U, c.V, c.W, c.P, c.rhs), want[i]):
            assert np.array_equal(a.download(), b), (i, _sizes(len(cases))[i], lab)


@pytest.mark.parametrize("n,precision,sweeps,solve_only", [(72, dfp.DFP_FP32_REFINE, 8, False),
                                                           (72, dfp.DFP_FP64, None, True),
                                                           (36, dfp.DFP_FP64, None, False),
                                                           (36, dfp.DFP_FP32_REFINE, 1, True)])
@pytest.mark.parametrize("graphs", [False, True])
def test_diverse_batch_equals_single_plans(n, precision, sweeps, solve_only, graphs):
    print(f"{n} cases, precision {precision}, {sweeps} sweeps, solve only {solve_only}, graphs {graphs}", flush=True)
    cases, start, want = _cases(n, precision, sweeps, solve_only)
    batch = Batch(max_cases=n, graphs=graphs)
    for _ in range(3 if graphs else 1):  # with graphs: captured, then replayed
        _run(batch, range(n), cases, start, want, solve_only)
    batch.close()
    for c in cases:
        c.plan.close()


def test_graphs_of_alternating_sets_of_sizes():
    """Sets of sizes in turn, each captured, then replayed, another set between: every call equals the single plans'
    bits."""
    print("graphs over alternating sets of sizes", flush=True)
    cases, start, want = _cases(12)
    batch = Batch(max_cases=12, graphs=True)
    for call in range(8):
        _run(batch, range(12) if call == 5 else range(call % 2, 12, 2), cases, start, want)
    batch.close()
    for c in cases:
        c.plan.close()
