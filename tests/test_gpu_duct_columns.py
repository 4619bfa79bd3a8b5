"""The duct's y solve with the columns in registers: row counts at the edges of
a chunk, of each column grouping (16, 8 and 4 modes per workgroup) and of the
lane-per-column sweep beyond them, mode counts that leave the last group
partial, against the C oracle."""
from __future__ import annotations

import pytest

import dfp
from _cases import fields, oracle_project, rel_linf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nym,nzm", [(1, 5), (15, 3), (16, 16), (17, 17), (255, 7), (256, 18), (257, 9), (512, 5),
                                     (513, 6), (1024, 4), (1025, 5)])
def test_duct_columns_match_oracle(nym, nzm):
    print(f"duct columns of {nym} rows, {nzm} modes", flush=True)
    g = dfp.duct_grid(4, nym, nzm, 1.0, 0.7)
    U, V, W, P, rhs = fields(g, nym + nzm, 0.1)
    o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    oracle_project(g, *o, 1e-3, 0.75, save_p=True)
    plan = dfp.Plan(g)
    d = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    plan.project(d[0], d[1], d[2], d[4], d[3], 1e-3, 0.75, save_p=True)
    plan.close()
    for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
        assert rel_linf(a, b) <= 1e-12, lab
