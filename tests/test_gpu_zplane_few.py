"""The library's choice of the z kernel where there are few sub-planes.
Periodic y: tall planes of short rows keep the LDS-resident kernel below 10
planes of 128 rows and 40 of 256.  Walls: a few planes of very few short rows
keep the streaming kernel.  Registers take the rest, and a z split asked for
takes registers wherever they fit.  Each side of the line against the C
oracle, and the shape reported makes the same plan."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from _cases import fields, make_grid, oracle_project, rel_linf

pytestmark = pytest.mark.gpu

DT, C3 = 1e-3, 0.75


def _project(g, tuning, host):
    plan = dfp.Plan(g, tuning=tuning)
    d = [a.copy(order="F") for a in host]
    plan.project(d[0], d[1], d[2], d[4], d[3], DT, C3, save_p=True)
    shape = plan.tuning
    plan.close()
    return shape, d


@pytest.mark.parametrize("nxp,nyp,nzp,planes", [(16, 128, 8, False), (18, 128, 8, True), (16, 64, 8, True),
                                                (72, 256, 8, False), (96, 256, 8, True), (36, 256, 16, False),
                                                (48, 256, 16, True), (8, 256, 128, True), (8, 128, 12, False)])
def test_few_planes_of_a_periodic_y(nxp, nyp, nzp, planes):
    print(f"periodic y {nxp}x{nyp + 1}x{nzp}", flush=True)
    g = dfp.periodic_y_grid(nxp, nyp + 1, nzp)
    host = fields(g, nyp + nzp, 0.1)
    o = [a.copy(order="F") for a in host]
    oracle_project(g, *o, DT, C3, save_p=True)
    shape, d = _project(g, None, host)
    assert shape[3] == (0 if planes else 2)
    for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
        assert rel_linf(a, b) <= 1e-12, lab
    again, e = _project(g, shape, host)
    assert again == shape and all(np.array_equal(a, b) for a, b in zip(d, e))


@pytest.mark.parametrize("nxp,nym,nzp,planes", [(16, 12, 32, False), (16, 13, 32, True), (32, 6, 64, False),
                                                (32, 7, 64, True), (64, 6, 64, False), (72, 6, 64, True),
                                                (16, 1, 128, True), (48, 1, 16, False)])
def test_few_planes_of_few_rows_between_walls(nxp, nym, nzp, planes):
    print(f"channel {nxp}x{nym}x{nzp}", flush=True)
    g = make_grid(nxp, nym, nzp, 1.5)
    host = fields(g, nym + nzp, 0.1)
    o = [a.copy(order="F") for a in host]
    oracle_project(g, *o, DT, C3, save_p=True)
    shape, d = _project(g, None, host)
    assert shape[3] == (0 if planes else 1)
    for lab, a, b in zip(("U", "V", "W", "P", "phi"), d, o):
        assert rel_linf(a, b) <= 1e-12, lab
    again, e = _project(g, shape, host)
    assert again == shape and all(np.array_equal(a, b) for a, b in zip(d, e))
    assert _project(g, (shape[0], 0, 0, 0), host)[0][3] == 0
