"""Batches of few, about as many, and more LU-SGS bands than the chip has compute units (256), and
than twice as many, where the band launches take other forms: every case equals its run alone, bit
for bit.  Bands of one row make many of them from small grids."""
import numpy as np
import pytest

from minismac_amd._abi import SMAC_FP32_LHS, SMAC_FP64
from minismac_amd.case import naca_case
from minismac_amd.solver import Batch, Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iturb", [0, 1])
@pytest.mark.parametrize("precision", [SMAC_FP64, SMAC_FP32_LHS])
@pytest.mark.parametrize("n", [1, 2, 4, 5, 9])
def test_many_bands_equal_alone(n, precision, iturb):
    # 61, 122, 244, 305 and 549 bands; with one row a band the scalar system has as many
    case = naca_case(63, 61, impsch=2, alpha=3.0, reynum=1e4, wall_spacing=1e-3, dtau=0.01, iturb=iturb,
                     precision=precision)
    opts = {"lusgs_rows": 1}
    with Solver(case, options=opts) as s:
        s.run(4)
        ref = s.get_state()
    solvers = [Solver(case, options=opts) for _ in range(n)]
    Batch(solvers).run(4)
    for s in solvers:
        for a, b in zip(s.get_state(), ref):
            assert np.array_equal(a, b)
        s.close()


@pytest.mark.parametrize("precision", [SMAC_FP64, SMAC_FP32_LHS])
@pytest.mark.parametrize("km", [119, 121, 521])
def test_one_case_of_many_bands(km, precision):
    # bands of one row, beside the SA's: 238, 242 and 1042 of both systems
    case = naca_case(63, km, impsch=2, alpha=3.0, reynum=1e4, wall_spacing=1e-3, dtau=0.001,
                     precision=precision)
    out = []
    for rows in (1, 64):
        with Solver(case, options={"lusgs_rows": rows}) as s:
            s.run(4)
            out.append(s.get_state())
    for a, b in zip(*out):
        assert np.array_equal(a, b)
