"""The library's choice of the z kernel for a periodic y where there are few
sub-planes: tall planes of short rows keep the LDS-resident kernel below 10
planes of 128 rows and 40 of 256, registers take the rest; a z split asked for
takes registers wherever they fit.  Each side of the line against the C
oracle, and the shape reported makes the same plan."""
from __future__ import annotations

import numpy as np
import pytest

import dfp
from _cases import fields, oracle_project, rel_linf

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
