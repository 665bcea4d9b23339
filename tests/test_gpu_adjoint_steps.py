"""The transposed line sweeps' fused steps for every mix of directions: with both, the terms of
the last eta step reach the xi sweeps on the way back to the natural layout; with one, the
first step of a colour starts the sum.  <P v, w> = <v, P^T w>, on line lengths at one wave's
end."""
import numpy as np
import pytest

from minismac_amd._abi import SMAC_ORDER_ZEBRA
from minismac_amd.case import naca_case
from minismac_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jm,km", [(81, 17), (97, 64), (101, 65)])
@pytest.mark.parametrize("njsp,nksp", [(1, 0), (0, 1), (2, 1), (1, 3)])
def test_update_and_its_transpose_agree(jm, km, njsp, nksp):
    case = naca_case(jm, km, impsch=1, line_order=SMAC_ORDER_ZEBRA, iturb=0, reynum=1000.0,
                     dtau=1.0, underr=0.8, wall_spacing=1e-3, njsp=njsp, nksp=nksp)
    rng = np.random.default_rng(jm + 10 * njsp + nksp)
    with Solver(case) as g:
        g.run(5)
        g.adjoint((), maxit=2, tol=1e-3, check=False)
        v, w = (np.asfortranarray(a) for a in rng.standard_normal((2, jm, km, 3)))
        pv, ptw = g.adjoint_apply(3, v), g.adjoint_apply(2, w)
    assert np.isfinite(pv).all() and np.isfinite(ptw).all()
    # each side's solves are accurate to a few hundred roundings of their result's size
    assert abs(np.vdot(pv, w) - np.vdot(v, ptw)) <= 1e-11 * np.linalg.norm(pv) * np.linalg.norm(w)
