"""The line factorisation where its grouping changes: one line per workgroup up to 1024 waves,
four lines (16-point chunks) beyond, on grids whose short lines end on, before and after a
chunk, against the oracle and through the identity <P v, w> = <v, P^T w> (P takes the twisted
factorisation of the blocks, P^T the plain one of the transposed blocks)."""
import numpy as np
import pytest

import pyoracle
from minismac_amd._abi import SMAC_ORDER_ZEBRA
from minismac_amd.case import naca_case
from minismac_amd.solver import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jm,km", [(1025, 17), (1031, 16), (1041, 33)])
def test_scan_passes_track_the_oracle(jm, km):
    case = naca_case(jm, km, impsch=1, alpha=2.0, reynum=1.0e6)
    o = pyoracle.Oracle(case)
    with Solver(case, options={"lr_solve": 1}) as g:
        for _ in range(3):
            gs, os_ = g.step(), o.step()
        q, _, _ = g.get_state()
    assert gs["rhsnorm"] == pytest.approx(os_["rhsnorm"], rel=1e-10)
    qo = o.array("q")
    assert np.abs(q - qo).max() <= 1e-10 * np.abs(qo).max()


@pytest.mark.parametrize("jm,km", [(511, 15), (513, 17), (601, 32), (641, 34), (1033, 65)])
def test_zebra_update_and_its_transpose_agree(jm, km):
    case = naca_case(jm, km, impsch=1, line_order=SMAC_ORDER_ZEBRA, iturb=0, reynum=1000.0,
                     dtau=1.0, underr=0.8, wall_spacing=1e-3)
    rng = np.random.default_rng(jm)
    with Solver(case) as g:
        g.run(20)
        g.adjoint((), maxit=2, tol=1e-3, check=False)
        v, w = rng.standard_normal((2, jm, km, 3))
        v, w = np.asfortranarray(v), np.asfortranarray(w)
        pv, ptw = g.adjoint_apply(3, v), g.adjoint_apply(2, w)
    assert np.isfinite(pv).all() and np.isfinite(ptw).all()
    assert abs(np.vdot(pv, w) - np.vdot(v, ptw)) <= 1e-11 * np.linalg.norm(pv) * np.linalg.norm(w)
