"""What the z eigenbasis leaves in the divergence of a duct's projection, for
wall cells so thin that the rounding of their coordinates shows: the general
bar, max|div u| <= 1e-12 max|u| / min spacing, whichever eigenvectors the plan
takes (even and odd ones up to a rounding of 1e-13 of a width, dense beyond)."""
from __future__ import annotations

import numpy as np
import pytest

import dfp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nzm,alpha_z", [(256, 2.0), (256, 3.2), (400, 3.2), (512, 3.2), (768, 0.0), (768, 3.2),
                                         (1000, 3.2)])
@pytest.mark.parametrize("make", [dfp.duct_grid, dfp.zwall_periodic_y_grid])
def test_projection_of_thin_wall_cells_is_divergence_free(make, nzm, alpha_z):
    print(f"{make.__name__} {nzm} cells, stretching {alpha_z}", flush=True)
    g = make(8, 33, nzm, 1.5, alpha_z) if make is dfp.duct_grid else make(8, 33, nzm, alpha_z)
    plan = dfp.Plan(g)
    F = [dfp.DeviceArray(s) for s in (g.shape_u, g.shape_v, g.shape_w)]
    rhs = dfp.DeviceArray(g.shape_rhs, zero=True)
    plan.synth(*F, 5, 0.2)
    alphas = [None] * 3
    if make is dfp.duct_grid:
        alphas = [dfp.DeviceArray((s[0], 2, s[2]), zero=True) for s in (g.shape_u, g.shape_v, g.shape_w)]
    plan.apply_bc(*F, *alphas)
    top = max(float(np.abs(f.download()).max()) for f in F)
    plan.project(*F, rhs, None, 1e-3, 0.75)
    plan.apply_bc(*F, *alphas)
    spacing = min(float(np.diff(g.z).min()), float(np.diff(g.y).min()), g.dx)
    div = plan.max_divergence(*F)
    plan.close()
    print(f"max|div u| spacing / max|u| = {div * spacing / top:.2e}", flush=True)
    assert div <= 1e-12 * top / spacing
