"""The substage writes its ghosts with the update and the correction: one
substage against the oracle's sequence (update, boundary conditions,
projection, boundary conditions), and bit for bit against the boundary-condition
entry point applied to the result once more (every ghost is a function of the
interior, so it must change nothing).  Grids: each flow, the fewest cells per
direction, several wavefronts per row."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from oracle import ref_c
from _cases import rel_linf
from test_gpu_step import DT, RK_COEF, _dev, _inputs

pytestmark = pytest.mark.gpu

GRIDS = {
    "channel_2x2x1": lambda: dfp.channel_grid(2, 2, 1, 1.0),
    "channel_4x3x2": lambda: dfp.channel_grid(4, 3, 2, 1.0),
    "channel_8x1x4": lambda: dfp.channel_grid(8, 1, 4, 1.0),
    "channel_162x9x12": lambda: dfp.channel_grid(162, 9, 12, 2.0),
    "box_4x2x2": lambda: dfp.periodic_y_grid(4, 2, 2),
    "box_2x3x1": lambda: dfp.periodic_y_grid(2, 3, 1),
    "box_24x10x9": lambda: dfp.periodic_y_grid(24, 10, 9),
    "duct_4x2x2": lambda: dfp.duct_grid(4, 2, 2, 1.0, 1.0),
    "duct_4x3x1": lambda: dfp.duct_grid(4, 3, 1, 1.0),
    "duct_18x7x11": lambda: dfp.duct_grid(18, 7, 11, 1.5, 1.0),
    "zwall_4x3x2": lambda: dfp.zwall_periodic_y_grid(4, 3, 2),
    "zwall_12x9x7": lambda: dfp.zwall_periodic_y_grid(12, 9, 7, 1.5),
}


@pytest.mark.parametrize("name", list(GRIDS))
@pytest.mark.parametrize("stage", [1, 2, 3])
def test_substep_ghosts(name, stage):
    print(f"substep {name} stage {stage}", flush=True)
    g = GRIDS[name]()
    F3, Fo, F, al = _inputs(g, 40 + stage)
    P, rhs = np.zeros(g.shape_p, order="F"), np.zeros(g.shape_rhs, order="F")
    c = RK_COEF[stage - 1][stage - 1]
    op = ref_c.CProjection(g)
    o = [a.copy(order="F") for a in (*F3, P, rhs)]
    op.rk_update(stage, *o[:3], *Fo, *F, RK_COEF[stage - 1], DT)
    op.apply_boundary_conditions(*o[:3], *al)
    op.compute_projection_step(*o[:3], o[4], o[3], DT, c)
    op.apply_boundary_conditions(*o[:3], *al)
    op.close()
    plan = dfp.Plan(g)
    d = [_dev(a) for a in (*F3, P, rhs)]
    ald = [_dev(a) for a in al]
    plan.substep(stage, *d[:3], *[_dev(a) for a in Fo], *[[_dev(x) for x in f] for f in F], RK_COEF[stage - 1], *ald,
                 d[4], d[3], DT, save_p=True)
    got = [x.download() for x in d]
    for lab, x, y in zip(("U", "V", "W", "P", "phi"), got, o):
        assert rel_linf(x, y) <= 1e-12, (lab, rel_linf(x, y))
    plan.apply_bc(*d[:3], *ald)
    for lab, x, y in zip("UVW", d, got):
        assert np.array_equal(x.download(), y), lab
    plan.close()
