"""The z kernel that holds a sub-plane in registers (the library's choice
where it fits): every row length, one and two passes per thread, a single
chunk, a partial last chunk, the largest plane of each form and the first one
beyond it (the streaming kernel), several planes per workgroup with a partial
last one, FP64 and FP32+refine.

FP64: the parity bar against the C oracle, and against the streaming kernel
on the same input: the two run the same recurrence with the chunk carries
associated differently, a round-off that grows with the length of the chain,
1e-13 at 40 rows (the fused kernel's bar) times nym/40.  FP32+refine: no
further from the oracle than the streaming kernel (one sweep leaves the error
of the FP32 form itself, about 1e-11 on the tallest of these grids).  Where
that kernel factors the row alike, the two round alike; where it transforms
in stages (18, 27, 54, 81, 108 modes), they are two samples of the same FP32
rounding error, equal in the mean over seeds and allowed a factor 3 here."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from _cases import fields, make_grid, oracle_project, rel_linf

pytestmark = pytest.mark.gpu

DT, C3 = 1e-3, 0.75
# row length: rows per pass, threads of the two-pass form
LENGTHS = {8: (8, 768), 12: (8, 768), 16: (8, 768), 18: (8, 512), 24: (8, 768), 27: (9, 512), 32: (8, 768),
           36: (8, 512), 48: (8, 768), 54: (9, 512), 64: (8, 768), 72: (8, 768), 81: (9, 512), 96: (8, 512),
           108: (9, 512), 128: (8, 512)}


def _rows(n):
    """nym at the edges of the forms of row length n (at most 400 rows)."""
    br, wide = LENGTHS[n]
    one, two = (384 // n) * br, (wide // n) * 2 * br
    return sorted({1, br - 1, br + 1, one, one + 1, two - 1, two, two + 1} & set(range(1, 401)))


@pytest.mark.parametrize("n", list(LENGTHS))
def test_register_planes_match_oracle_and_streaming_kernel(n):
    br, wide = LENGTHS[n]
    for nym in _rows(n):
        print(f"rows of {n} modes, nym {nym}", flush=True)
        g = make_grid(6, nym, n, 1.5)
        U, V, W, P, rhs = fields(g, n + nym, 0.1)
        o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
        oracle_project(g, *o, DT, C3, save_p=True)
        for prec in (dfp.DFP_FP64, dfp.DFP_FP32_REFINE):
            outs, errs = [], []
            for tuning in ((1, 0, 0, 0), (1, 0, 0, 1)):
                plan = dfp.Plan(g, precision=prec, tuning=tuning)
                fits = nym <= (wide // n) * 2 * br
                assert plan.tuning[3] == (0 if fits and tuning[3] == 0 else 1)
                d = [a.copy(order="F") for a in (U, V, W, P, rhs)]
                plan.project(d[0], d[1], d[2], d[4], d[3], DT, C3, save_p=True)
                plan.close()
                outs.append(d)
                errs.append([rel_linf(a, b) for a, b in zip(d, o)])
            if prec == dfp.DFP_FP64:
                assert max(errs[0]) <= 1e-12, (nym, errs)
                assert max(rel_linf(a, b) for a, b in zip(*outs)) <= 1e-13 * max(1.0, nym / 40), nym
            else:
                slack = 3.0 if n in (18, 27, 54, 81, 108) else 1.1
                assert max(errs[0]) <= slack * max(errs[1]) + 1e-13, (nym, errs)


@pytest.mark.parametrize("nxp,nym,nzp,R", [(8, 24, 32, 4), (6, 10, 72, 9), (16, 17, 64, 2), (12, 5, 24, 1)])
def test_register_planes_several_per_workgroup(nxp, nym, nzp, R):
    """Sub-planes of a few threads share a workgroup; repeated runs give the same bits."""
    g = make_grid(nxp, nym, nzp, 1.7)
    U, V, W, P, rhs = fields(g, 11, 0.1)
    o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    oracle_project(g, *o, DT, C3, save_p=True)
    plan = dfp.Plan(g, tuning=(R, 0, 0, 0))
    first = None
    for _ in range(2):
        d = [a.copy(order="F") for a in (U, V, W, P, rhs)]
        plan.project(d[0], d[1], d[2], d[4], d[3], DT, C3, save_p=True)
        for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
            assert rel_linf(a, b) <= 1e-12, lab
        assert first is None or all(np.array_equal(a, b) for a, b in zip(d, first))
        first = d
    plan.close()
