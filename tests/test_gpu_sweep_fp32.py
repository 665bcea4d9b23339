"""The FP32-LHS LU-SGS sweeps, whose rows run in groups of four, each some steps behind the one
before, against the FP64 ones from the same state, at bands of one row, of parts of a group, of
whole groups, and cut off by the grid's last row, alone and in a batch.

A pass's dq differs by FP32's rounding (6e-8) of the operands and of the sums, which grow along
the sweeps by what the recurrence carries on: within 1e-4 of the largest dq, where a value taken
from a wrong point, component or step differs by about the value itself."""
import numpy as np
import pytest

from minismac_amd._abi import SMAC_FP32_LHS, SMAC_FP64
from minismac_amd.case import naca_case
from minismac_amd.solver import Batch, Solver

pytestmark = pytest.mark.gpu


def _case(jm, km, precision):
    return naca_case(jm, km, impsch=2, alpha=3.0, reynum=1e3, wall_spacing=1e-3, dtau=0.1, iturb=0,
                     precision=precision)


def _dq(case, rows, passes=2):
    with Solver(case, options={"lusgs_rows": rows}) as s:
        for _ in range(passes):
            s.step()
        return s.array("dq")


@pytest.mark.parametrize("jm,km,rows", [(11, 5, 16), (21, 8, 16), (33, 12, 16), (35, 16, 16),
                                        (41, 17, 16), (61, 20, 16), (63, 33, 16), (129, 61, 16),
                                        (41, 17, 1), (41, 18, 3), (61, 21, 4), (61, 29, 5),
                                        (61, 33, 9), (61, 40, 13)])
def test_fp32_sweeps_follow_fp64(jm, km, rows):
    a, b = (_dq(_case(jm, km, p), rows) for p in (SMAC_FP64, SMAC_FP32_LHS))
    assert np.all(np.isfinite(b))
    assert np.abs(b - a).max() <= 1e-4 * np.abs(a).max()


def test_fp32_sweeps_in_a_batch_equal_alone():
    cases = [_case(j, k, SMAC_FP32_LHS) for j, k in ((41, 17), (63, 33), (129, 61))]
    alone = []
    for c in cases:
        with Solver(c) as s:
            s.run(4)
            alone.append(s.get_state()[0])
    solvers = [Solver(c) for c in cases]
    Batch(solvers).run(4)
    for s, q in zip(solvers, alone):
        assert np.array_equal(s.get_state()[0], q)
