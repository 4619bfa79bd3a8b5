"""z rows of fewer than 8 modes under more than 256 y rows: a row group of the
streaming z kernel holds no more rows than its workgroup has threads to stage
their coefficients, against the C oracle (FP64 and FP32+refine, whose own
error after three sweeps stays below the parity bar on these grids)."""
from __future__ import annotations

import pytest

import dfp
from _cases import fields, make_grid, oracle_project, rel_linf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nym,nzp", [(257, 1), (300, 4), (513, 6), (300, 8)])
def test_short_rows_tall_planes(nym, nzp):
    print(f"rows of {nzp} points, {nym} y rows", flush=True)
    g = make_grid(8, nym, nzp, 1.2)
    U, V, W, P, rhs = fields(g, nym, 0.1)
    o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    oracle_project(g, *o, 1e-3, 0.75, save_p=True)
    for prec, sweeps, tol in ((dfp.DFP_FP64, None, 1e-12), (dfp.DFP_FP32_REFINE, 3, 1e-11)):
        plan = dfp.Plan(g, precision=prec, sweeps=sweeps)
        d = [a.copy(order="F") for a in (U, V, W, P, rhs)]
        plan.project(d[0], d[1], d[2], d[4], d[3], 1e-3, 0.75, save_p=True)
        plan.close()
        for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
            assert rel_linf(a, b) <= tol, (prec, lab)
