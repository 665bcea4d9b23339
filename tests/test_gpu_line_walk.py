"""Line relaxation in the reference's line order with every line solved by scans, at lines that end
on, before and after a wave's 64 points and the 128 (FP64) and 256 (FP32) up to which a second
group of waves forms the scans' matrices, against the sequential form (the oracle's bits), one pass.

The bound follows from the system: rounding its blocks once to FP32 moves the oracle's dq by `sens`.
A pass rounds some 250 times on the way to a value (four sweeps of two scans, about eight steps of
four operations each), so it is held to 1000 sens, and in FP64 to 2^-29 of that.  A value taken from a
wrong point, step or line moves dq by 3e-3 to 7 of its largest, where the line couples its points."""
import numpy as np
import pytest

import pyoracle
from minismac_amd._abi import SMAC_FP32_LHS, SMAC_FP64, SMAC_ORDER_REFERENCE, SMAC_ORDER_ZEBRA
from minismac_amd.case import naca_case
from minismac_amd.solver import Solver

pytestmark = pytest.mark.gpu

BLOCKS = ("btc", "bjm", "bjp", "bkm", "bkp")


def _case(jm, km, precision):
    return naca_case(jm, km, impsch=1, alpha=3.0, reynum=1e3, wall_spacing=1e-3, dtau=0.1, underr=0.3,
                     iturb=0, precision=precision)


def _dq(case, scan):
    with Solver(case, options={"lr_solve": 1} if scan else {}) as s:
        s.step()
        return s.array("dq")


def _sens(case):
    o = pyoracle.Oracle(case)
    q = o.array("q").copy(order="F")
    o.step()
    out = []
    for t in (np.float64, np.float32):
        blocks = (np.asfortranarray(o.array("lhs_" + b).astype(t).astype(np.float64)) for b in BLOCKS)
        dq = np.zeros_like(q, order="F")
        pyoracle.lrelax(case.params, q, dq, np.asfortranarray(o.array("s").copy()), *blocks,
                        wake_pairs=case.wake_pairs())
        out.append(dq)
    return np.abs(out[1] - out[0]).max()


@pytest.mark.parametrize("jm,km", [(11, 5), (63, 64), (65, 65), (21, 63), (127, 128), (129, 9), (21, 129),
                                   (255, 7), (257, 12), (31, 256), (31, 257)])
def test_walk_follows_the_sequential_form(jm, km):
    case = _case(jm, km, SMAC_FP64)
    ref, tol = _dq(case, False), 1000 * _sens(case)
    assert np.abs(_dq(case, True) - ref).max() <= tol * 2.0 ** -29
    assert np.abs(_dq(_case(jm, km, SMAC_FP32_LHS), True) - ref).max() <= tol


@pytest.mark.parametrize("precision", [SMAC_FP64, SMAC_FP32_LHS])
@pytest.mark.parametrize("order", [SMAC_ORDER_REFERENCE, SMAC_ORDER_ZEBRA])
def test_cut_rows_of_the_rhs(order, precision):
    """After a pass whose last sweeps are eta ones the natural right-hand side holds the injected
    values in the cut's points, as dq does, and the assembled ones everywhere else."""
    case = naca_case(63, 17, impsch=1, alpha=3.0, reynum=1e3, wall_spacing=1e-3, dtau=0.1, underr=0.3,
                     iturb=0, precision=precision, line_order=order)
    o = pyoracle.Oracle(case)
    o.step()
    with Solver(case, options={"lr_solve": 1}) as g:
        g.step()
        s, dq = g.array("s"), g.array("dq")
    cut = np.unique(case.wake_pairs()[:, 0]) - 1
    assert np.array_equal(s[cut, 0], dq[cut, 0])
    rest = np.ones(s.shape[:2], bool)
    rest[cut, 0] = False
    assert np.array_equal(s[rest], o.array("s")[rest])
