"""The periodic-y z/y kernel with its sub-planes in registers (the library's
choice where it takes the shape): every row length and column split, planes
that share a workgroup with a partial last one, against the C oracle; lengths
beside them keep the LDS kernel."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from _cases import fields, oracle_project, rel_linf

pytestmark = pytest.mark.gpu

SHAPES = [(n, nyp) for n in (8, 12, 16, 24, 32, 48, 64) for nyp in (16, 32, 64, 128, 256)
          if n * {16: 2, 32: 4, 64: 8, 128: 8, 256: 16}[nyp] <= 512]


def _run(nxp, nym, nzp, tuning, planes):
    g = dfp.periodic_y_grid(nxp, nym, nzp)
    print(f"periodic y {nxp}x{nym}x{nzp} tuning {tuning}", flush=True)
    U, V, W, P, rhs = fields(g, nym + nzp, 0.1)
    o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    oracle_project(g, *o, 1e-3, 0.75, save_p=True)
    plan = dfp.Plan(g, tuning=tuning)
    assert plan.tuning[3] == (0 if planes else 2)
    d = [a.copy(order="F") for a in (U, V, W, P, rhs)]
    plan.project(d[0], d[1], d[2], d[4], d[3], 1e-3, 0.75, save_p=True)
    plan.close()
    for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
        assert rel_linf(a, b) <= 1e-12, lab
    assert np.array_equal(d[4][:, nym - 1, :], d[4][:, 0, :])


@pytest.mark.parametrize("n,nyp", SHAPES)
def test_register_planes_match_oracle(n, nyp):
    _run(6, nyp + 1, n, (1, 0, 0, 0), True)


@pytest.mark.parametrize("nxp,nym,nzp,R", [(8, 17, 32, 4), (6, 17, 72, 9), (16, 33, 16, 2)])
def test_several_planes_per_workgroup(nxp, nym, nzp, R):
    _run(nxp, nym, nzp, (R, 0, 0, 0), True)


@pytest.mark.parametrize("nym,nzp", [(9, 8), (28, 8), (17, 18), (257, 6)])
def test_other_lengths_keep_the_lds_kernel(nym, nzp):
    _run(6, nym, nzp, (1, 0, 0, 0), False)
