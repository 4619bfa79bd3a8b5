"""The z eigenbasis transforms of a z grid symmetric about its middle (even and
odd eigenmodes apart) and of one that is not (the dense transforms), against
the C oracle: odd and even cell counts around the tiles of 32 columns and the
stages of 16, partial row tiles, the duct and the z walls with a periodic y."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from dfp.grid import _centres
from _cases import fields, oracle_project, rel_linf

pytestmark = pytest.mark.gpu


def _skewed(g):
    """The grid with its z faces moved by up to a tenth of a cell, no longer symmetric."""
    r = np.random.default_rng(5).uniform(-0.1, 0.1, g.z.size)
    r[0] = r[-1] = 0.0
    g.z = g.z + r * np.min(np.diff(g.z))
    g.zg = _centres(g.z)
    g.dz = float(np.min(np.diff(g.zg)))
    return g


@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("nym,nzm", [(9, 1), (5, 2), (7, 3), (65, 16), (64, 31), (66, 32), (9, 33), (17, 63), (9, 64),
                                     (129, 65), (9, 131)])
def test_z_eigenbasis_matches_oracle(nym, nzm, skew):
    for make in (lambda: dfp.duct_grid(6, nym, nzm, 1.3, 1.1),
                 lambda: dfp.zwall_periodic_y_grid(6, {5: 5, 7: 7, 64: 55, 65: 65, 66: 73, 129: 129}.get(nym, nym), nzm,
                                                   0.9)):
        g = make()
        if skew and nzm > 1:
            g = _skewed(g)
        print(f"z eigenbasis {g.nym} rows, {nzm} cells, y_bc {g.y_bc_type}, skew {skew}", flush=True)
        U, V, W, P, rhs = fields(g, nym + nzm, 0.1)
        o = [a.copy(order="F") for a in (U, V, W, P, rhs)]
        oracle_project(g, *o, 1e-3, 0.75, save_p=True)
        plan = dfp.Plan(g)
        d = [a.copy(order="F") for a in (U, V, W, P, rhs)]
        plan.project(d[0], d[1], d[2], d[4], d[3], 1e-3, 0.75, save_p=True)
        plan.close()
        for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
            assert rel_linf(a, b) <= 1e-12, (lab, g.y_bc_type)
