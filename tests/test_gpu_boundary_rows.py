"""Boundary rows, residual norms and wall forces against the oracle, bit for bit, at grids whose
far field and outflow end on, before and after a workgroup's 64 points, and whose walls fill none,
one or more chunks of 448 faces, with and without the viscous forces."""
import numpy as np
import pytest

import pyoracle
from minismac_amd.case import naca_case
from minismac_amd.solver import Solver

pytestmark = pytest.mark.gpu

EXACT = ("resmax", "jres", "kres", "divmax", "cl", "cd", "cm", "fxp", "fyp", "fxs", "fys", "fmom")


@pytest.mark.parametrize("jm,km,ivis", [(11, 5, 1), (63, 66, 1), (65, 64, 0), (67, 65, 1), (679, 6, 1),
                                        (681, 5, 0), (683, 5, 1), (1361, 5, 1), (1365, 5, 0),
                                        (2047, 5, 1)])
def test_rows_and_forces_match_oracle(jm, km, ivis):
    # a short pseudo-time step: these grids are too coarse for the default to stay finite
    case = naca_case(jm, km, impsch=2, alpha=3.0, reynum=1e5, wall_spacing=1e-4, dtau=1e-3, ivis=ivis,
                     iturb=0)
    o = pyoracle.Oracle(case)
    with Solver(case, keep_lhs=True) as g:
        for _ in range(3):
            gs, os_ = g.step(), o.step()
            for k in EXACT:
                assert gs[k] == os_[k], k
            assert gs["rhsnorm"] == pytest.approx(os_["rhsnorm"], rel=1e-13, abs=0)
        for name in ("btc", "bjm", "bjp", "bkm", "bkp"):
            assert np.array_equal(g.array(name), o.array("lhs_" + name)), name
        assert np.array_equal(g.get_state()[0], o.array("q"))
