"""The FP64 (0,0)-mode solve of the FP32+refine form on its own: a right-hand
side that depends on y only leaves every other FP32 mode exactly zero (lengths
that are powers of two), so phi is the mean solve.  Against the FP64 plan,
whose z kernel runs the same pinned recurrence: row counts around a wave, the
lanes' runs and the staging chunk.  Bar: 1e-13 at 40 rows, growing with the
length of the chain (carries associated differently)."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from _cases import make_grid, rel_linf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nym", [1, 2, 63, 64, 65, 129, 1023, 1024, 1025, 2500])
def test_mean_solve_matches_fp64(nym):
    print(f"mean solve, {nym} rows", flush=True)
    g = make_grid(8, nym, 4, 1.2)
    f = np.random.default_rng(nym).standard_normal(nym)
    out = []
    for prec in (dfp.DFP_FP64, dfp.DFP_FP32_REFINE):
        rhs = np.zeros(g.shape_rhs, order="F")
        rhs[:8, :, :4] = f[None, :, None]
        plan = dfp.Plan(g, precision=prec, sweeps=0 if prec else None)
        plan.solve(rhs)
        plan.close()
        out.append(rhs)
    assert rel_linf(out[1], out[0]) <= 1e-13 * max(1.0, nym / 40)
