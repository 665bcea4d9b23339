"""Adjoints with the LU-SGS preconditioner on grids of so many rows that its two solves run one
after the other (more than 1920) and of fewer: the residual each solve reports is that of the
solution it leaves."""
import numpy as np
import pytest

from minismac_amd.case import naca_case
from minismac_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("km", [1905, 1937])
def test_both_solves_leave_their_solutions(km):
    case = naca_case(11, km, impsch=2, alpha=2.0, reynum=100.0, wall_spacing=1e-2, dtau=1e-3, iturb=0)
    with Solver(case) as s:
        s.run(2)
        st = s.adjoint(maxit=6, tol=1e-14, check=False)[2]
        for o, name in enumerate(("cl", "cd")):
            g, lam = s.array("adj_g" + name), s.array("adj_lam_" + name)
            assert st["iters"][o] == 6 and np.all(np.isfinite(lam)) and np.abs(lam).max() > 0
            r = np.linalg.norm(g - s.adjoint_apply(1, lam)) / np.linalg.norm(g)
            assert r == pytest.approx(st["resid"][o], rel=1e-6)
