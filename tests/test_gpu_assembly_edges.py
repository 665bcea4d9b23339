"""The assembly against the oracle, bit for bit, on rows that end on, before and after a wave's
60 points, with one, two and four rows a wave and strips cut short at the last row, and the same
for a batch's cases (four rows a wave) against their own passes."""
import numpy as np
import pytest

import pyoracle
from minismac_amd.case import naca_case
from minismac_amd.solver import Batch, Solver

pytestmark = pytest.mark.gpu


def _case(jm, km, **kw):
    # a short pseudo-time step: these grids are too coarse for the default to stay finite
    return naca_case(jm, km, impsch=2, alpha=3.0, reynum=1e5, wall_spacing=1e-4, dtau=1e-3, **kw)


@pytest.mark.parametrize("jm,km,ivis", [(59, 5, 1), (61, 9, 1), (61, 8, 0), (119, 7, 1), (121, 6, 1),
                                        (181, 10, 1), (121, 691, 1), (61, 2051, 1)])
def test_assembly_matches_oracle(jm, km, ivis):
    case = _case(jm, km, ivis=ivis, iturb=0)
    o = pyoracle.Oracle(case)
    with Solver(case, keep_lhs=True) as g:
        for _ in range(3):
            gs, os_ = g.step(), o.step()
        for name in ("btc", "bjm", "bjp", "bkm", "bkp"):
            assert np.array_equal(g.array(name), o.array("lhs_" + name)), name
        assert np.array_equal(g.get_state()[0], o.array("q"))
    assert gs["rhsnorm"] == pytest.approx(os_["rhsnorm"], rel=1e-12)


def test_batch_assembly_matches_single():
    cases = [_case(j, k) for j, k in ((59, 9), (61, 10), (121, 11))]
    single = []
    for c in cases:
        with Solver(c) as s:
            s.run(4)
            single.append(s.get_state()[0])
    solvers = [Solver(c) for c in cases]
    Batch(solvers).run(4)
    for s, q in zip(solvers, single):
        assert np.array_equal(s.get_state()[0], q)
