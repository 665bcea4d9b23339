"""A batch whose cases have more boundary regions than one launch's table holds (16), with points
that regions of two tables share: the later region's rows win there, as in a case stepped alone
and in the oracle."""
import dataclasses

import numpy as np
import pytest

import pyoracle
from minismac_amd._abi import SMAC_FP32_LHS, SMAC_FP64
from minismac_amd.case import naca_case
from minismac_amd.solver import Batch, Solver

pytestmark = pytest.mark.gpu


def _split(case, pieces):
    """The far field in `pieces` regions that overlap in a point each and reach over the outflow's
    corners; the outflow again at the end, so that either order of two regions occurs."""
    jm = case.jmax
    ends = np.linspace(1, jm, pieces + 1).astype(int)
    far = [(25, 1, int(a), int(b), -1, -1) for a, b in zip(ends[:-1], ends[1:])]
    rest = [r for r in case.regions if r[0] not in (25, 31)]
    out = [r for r in case.regions if r[0] == 31]
    return dataclasses.replace(case, regions=out[:1] + rest + far + out[1:])


@pytest.mark.parametrize("precision", [SMAC_FP64, SMAC_FP32_LHS])
def test_regions_of_two_tables(precision):
    cases = [_split(naca_case(jm, km, impsch=2, alpha=3.0, reynum=1e5, wall_spacing=1e-4, dtau=1e-3,
                              precision=precision), n)
             for jm, km, n in ((63, 17, 12), (129, 33, 20), (239, 61, 37))]
    assert sum(len(c.regions) > 18 for c in cases) == 2
    alone = []
    for c in cases:
        with Solver(c) as s:
            s.run(4)
            alone.append((s.get_state(), s.array("s")))
    solvers = [Solver(c) for c in cases]
    Batch(solvers).run(4)
    for c, s, ((q, a, v), rows) in zip(cases, solvers, alone):
        qb, ab, vb = s.get_state()
        assert np.array_equal(qb, q) and np.array_equal(ab, a) and np.array_equal(vb, v)
        assert np.array_equal(s.array("s"), rows)
        if precision == SMAC_FP64:
            o = pyoracle.Oracle(c)
            for _ in range(4):
                o.step()
            assert np.array_equal(qb, o.array("q"))
        s.close()
