"""The FP32-LHS LU-SGS solve against the same arithmetic in numpy, bit for bit: the neighbour blocks
and the right-hand side premultiplied by the diagonal block's inverse, then at each point one fused
multiply-add a term, forward the j-neighbour's three terms before the k-neighbour's, backward the
other way round.  The blocks are the oracle's rounded to FP32, the points are taken hyperplane by
hyperplane, and nothing is known of bands, groups or hand-overs.

Every operation is a correctly rounded FP32 one on both sides, so the results are equal."""
import numpy as np
import pytest

import pyoracle
from minismac_amd._abi import SMAC_FP32_LHS
from minismac_amd.case import config_case, naca_case
from minismac_amd.solver import Solver

F = np.float32


def _fma(a, b, c):
    """a b + c, rounded once: the product is exact in FP64, its sum with c is rounded to odd there,
    which leaves the rounding to FP32 correct (53 bits are two more than twice 24)."""
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)
    even = (s.view(np.int64) & 1) == 0
    odd = np.nextafter(s, np.where(err > 0, np.inf, -np.inf))
    return np.where((err != 0) & even, odd, s).astype(F)


def _factor(t):
    f = [None] * 9
    one = F(1)
    f[0] = one / t[0]
    f[3] = t[3] * f[0]
    f[6] = t[6] * f[0]
    f[1] = t[1]
    f[4] = one / (t[4] - f[1] * f[3])
    f[7] = (t[7] - f[1] * f[6]) * f[4]
    f[2] = t[2]
    f[5] = t[5] - f[2] * f[3]
    f[8] = one / (t[8] - f[2] * f[6] - f[5] * f[7])
    return f


def _scaled(f, r):
    """D^-1 of a column r of three values"""
    z1 = r[0] * f[0]
    z2 = _fma(-f[1], z1, r[1]) * f[4]
    z3 = _fma(-f[5], z2, _fma(-f[2], z1, r[2])) * f[8]
    o1 = _fma(-f[7], z3, z2)
    return [_fma(-f[3], o1, _fma(-f[6], z3, z1)), o1, z3]


def _solve(case):
    o = pyoracle.Oracle(case)
    o.assemble()
    jm, km = case.jmax, case.kmax
    q, s = o.array("q"), o.array("s").astype(F)

    def block(name):
        b = o.array(name).reshape(jm, km, 9, order="F").astype(F)
        return [np.ascontiguousarray(b[:, :, m]) for m in range(9)]

    btc, bjm, bjp, bkm, bkp = (block(n) for n in ("btc", "bjm", "bjp", "bkm", "bkp"))
    f = _factor(btc)
    nb = []
    for b in (bjm, bkm, bjp, bkp):
        cols = [_scaled(f, b[3 * c:3 * c + 3]) for c in range(3)]
        nb.append(np.array(cols))                        # [n][c]: entry (c, n)
    lj, lk, uj, uk = nb
    x = np.array(_scaled(f, [s[:, :, c] for c in range(3)]))
    planes = [(h - k, k) for h in range(jm + km - 1) for k in (np.arange(max(0, h - jm + 1), min(km, h + 1)),)]

    def term(t, mat, at, has, frm):
        j, k = at
        for n in range(3):
            xn = x[n][frm]
            for c in range(3):
                t[c] = np.where(has, _fma(xn, -mat[n][c][j, k], t[c]), t[c])

    for j, k in planes:
        t = [x[c][j, k] for c in range(3)]
        term(t, lj, (j, k), j > 0, (np.maximum(j - 1, 0), k))
        term(t, lk, (j, k), k > 0, (j, np.maximum(k - 1, 0)))
        for c in range(3):
            x[c][j, k] = t[c]
    for j, k in reversed(planes):
        t = [x[c][j, k] for c in range(3)]
        term(t, uk, (j, k), k < km - 1, (j, np.minimum(k + 1, km - 1)))
        term(t, uj, (j, k), j < jm - 1, (np.minimum(j + 1, jm - 1), k))
        for c in range(3):
            x[c][j, k] = t[c]
    dq = np.moveaxis(x, 0, 2).astype(np.float64)
    for jt, jb in case.wake_pairs() - 1:
        snew = 0.5 * (q[jt, 1] + q[jb, 1])
        dsnew = 0.5 * (dq[jt, 1] + dq[jb, 1])
        dq[jt, 0] = snew + dsnew - q[jt, 0]
    return dq


def _case(jm, km):
    return naca_case(jm, km, impsch=2, alpha=3.0, reynum=1e3, wall_spacing=1e-3, dtau=0.1, iturb=0,
                     precision=SMAC_FP32_LHS)


def test_fma_is_rounded_once():
    rng = np.random.default_rng(5)
    a, b = (rng.uniform(1, 2, 2000).astype(F) for _ in range(2))
    c = (-(a.astype(np.float64) * b) * (1 + rng.choice([0, 2.0 ** -24, 2.0 ** -25, 1.0], 2000))).astype(F)
    from fractions import Fraction
    for x, y, z, got in zip(a, b, c, _fma(a, b, c)):
        want = Fraction(float(x)) * Fraction(float(y)) + Fraction(float(z))
        err = abs(Fraction(float(got)) - want)
        for other in (np.nextafter(got, F(np.inf)), np.nextafter(got, F(-np.inf))):
            assert err <= abs(Fraction(float(other)) - want)


@pytest.mark.gpu
@pytest.mark.parametrize("jm,km,rows", [(11, 5, 16), (21, 8, 16), (33, 12, 16), (35, 16, 16),
                                        (41, 17, 16), (61, 19, 16), (63, 33, 16), (129, 61, 16),
                                        (41, 18, 3), (61, 21, 4), (61, 33, 9), (61, 40, 13), (63, 50, 1)])
def test_fp32_solve_is_the_ordered_one(jm, km, rows):
    case = _case(jm, km)
    with Solver(case, options={"lusgs_rows": rows}) as s:
        s.step()
        assert np.array_equal(s.array("dq"), _solve(case))


@pytest.mark.gpu
def test_fp32_solve_at_945x241():
    case = config_case(1, impsch=2, precision=SMAC_FP32_LHS, iturb=0)
    with Solver(case) as s:
        s.step()
        assert np.array_equal(s.array("dq"), _solve(case))
