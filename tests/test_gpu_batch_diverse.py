"""Batches of many different sizes in one call: every stage then has many
launches (x kernels by z split and group of line lengths, z kernels by row
length), and the call takes them all.  Each case equals its own plan's bits."""
from __future__ import annotations

import pytest

import dfp
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


@pytest.mark.parametrize("n,precision,sweeps,solve_only", [(72, dfp.DFP_FP32_REFINE, 8, False),
                                                           (72, dfp.DFP_FP64, 0, True), (36, dfp.DFP_FP64, 0, False),
                                                           (36, dfp.DFP_FP32_REFINE, 1, True)])
@pytest.mark.parametrize("graphs", [False, True])
def test_diverse_batch_equals_single_plans(n, precision, sweeps, solve_only, graphs):
    import torch

    from dfp.batch import Batch, Case

    print(f"{n} cases, precision {precision}, {sweeps} sweeps, solve only {solve_only}, graphs {graphs}", flush=True)
    refine = sweeps if precision == dfp.DFP_FP32_REFINE else None
    cases, singles, start = [], [], []
    for i, (nxp, nym, nzp, R) in enumerate(_sizes(n)):
        g = make_grid(nxp, nym, nzp, 1.5)
        host = fields(g, i + 1, 0.1)
        one, two, new = ([torch.from_numpy(a.T.copy()).cuda() for a in host] for _ in range(3))
        plans = [dfp.Plan(g, precision=precision, sweeps=refine, tuning=(R, 0, 0, 0)) for _ in range(2)]
        for f in (one, two, new):
            if solve_only:
                plans[0].divergence(*f[:3], f[4])
        if solve_only:
            plans[0].solve(one[4], one[3], DT, C3, save_p=True)
        else:
            plans[0].project(*one[:3], one[4], one[3], DT, C3, save_p=True)
        plans[0].close()
        singles.append(one)
        start.append(new)
        U, V, W, P, rhs = two
        cases.append(Case(plans[1], U, V, W, rhs, P, DT, C3, save_p=True))
    batch = Batch(max_cases=n, graphs=graphs)
    for _ in range(3):  # with graphs: run, captured, replayed
        for c, f in zip(cases, start):
            for to, at in zip((c.U, c.V, c.W, c.P, c.rhs), f):
                to.copy_(at)
        torch.cuda.synchronize()
        batch.project(cases, solve_only=solve_only)
        for size, c, s in zip(_sizes(n), cases, singles):
            for lab, a, b in zip(("U", "V", "W", "P", "phi"), (c.U, c.V, c.W, c.P, c.rhs), s):
                assert torch.equal(a, b), (size, lab)
    batch.close()
    for c in cases:
        c.plan.close()


def test_graph_of_a_batch_is_captured_when_its_stage_list_comes_again():
    """Sets of sizes in turn, each run directly, then captured, then replayed, other sets between: every call equals
    the single plans' bits."""
    import torch

    from dfp.batch import Batch, Case

    print("graphs over alternating sets of sizes", flush=True)
    cases, start, want = [], [], []
    for i, (nxp, nym, nzp, R) in enumerate(_sizes(12)):
        g = make_grid(nxp, nym, nzp, 1.5)
        f = [torch.from_numpy(a.T.copy()).cuda() for a in fields(g, i + 1, 0.1)]
        start.append([a.clone() for a in f])
        one = [a.clone() for a in f]
        plan = dfp.Plan(g, tuning=(R, 0, 0, 0))
        plan.project(*one[:3], one[4], one[3], DT, C3, save_p=True)
        want.append(one)
        cases.append(Case(plan, *f[:3], f[4], f[3], DT, C3, save_p=True))
    batch = Batch(max_cases=12, graphs=True)
    for call in range(8):
        part = range(12)[call % 2::2] if call != 5 else range(12)
        for i in part:
            c = cases[i]
            for to, at in zip((c.U, c.V, c.W, c.P, c.rhs), start[i]):
                to.copy_(at)
        torch.cuda.synchronize()
        batch.project([cases[i] for i in part])
        for i in part:
            c = cases[i]
            for lab, a, b in zip(("U", "V", "W", "P", "phi"), (c.U, c.V, c.W, c.P, c.rhs), want[i]):
                assert torch.equal(a, b), (call, i, lab)
    batch.close()
    for c in cases:
        c.plan.close()
