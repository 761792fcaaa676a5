"""The FP64 kernels' own exponential against extended precision: on one
Black-Scholes step from a spot of 1 without rates, a call struck at 0 pays
exp(drift + std g) with the path's normal g, arguments of -30 to 14.  Within 0.9
of a unit in the last place: half a unit of the last addition, 0.17 of the factor
1 + d series rounded at |d| up to 0.35, 0.19 of the argument left after the
reduction; three in a hundred arguments would be off by more than 0.6 with one
rounding more.  Exact at 0."""
import numpy as np
import pytest

import compfinance_amd as cf

pytestmark = pytest.mark.gpu


def _fma(a, b, c):
    """a b + c of arrays in double, rounded once (Dekker's product and sums)."""
    def split(x):
        t = 134217729.0 * x
        return t - (t - x), x - (t - (t - x))

    p, (ah, al), (bh, bl) = a * b, split(a), split(b)
    err = ((ah * bh - p) + ah * bl + al * bh) + al * bl
    s = p + c
    t = s - p
    return s + (((p - (s - t)) + (c - t)) + err)


def test_exponentials_are_within_an_ulp(engine):
    assert np.finfo(np.longdouble).nmant >= 63
    n, vol, mat = 1 << 17, 2.0, 4.0
    g = cf.sobol_points(0, n, 1, cf.FP64, 1)[1][:, 0]
    num = cf.NumericalParam(numPath=n, precision=cf.FP64)
    got = cf.mcParallelSimul(cf.European(0.0, mat), cf.BlackScholes(1.0, vol, False, 0.0, 0.0), num=num).payoffs[:, 0]
    x = _fma(np.full(n, vol * np.sqrt(mat)), g, np.full(n, -0.5 * vol * vol * mat))
    ref = np.exp(x.astype(np.longdouble))
    ulps = np.abs((got.astype(np.longdouble) - ref) / np.spacing(ref.astype(np.float64))).astype(np.float64)
    assert ulps.max() <= 0.9, ulps.max()
    assert (ulps > 0.6).mean() <= 0.02, (ulps > 0.6).mean()


def test_exact_at_zero(engine):
    mdl = cf.Dupire(spot=1.0, spots=[0.5, 2.0], times=[1.0], vols=[[0.0], [0.0]], maxDt=1.0)
    num = cf.NumericalParam(numPath=64, precision=cf.FP64)
    assert np.all(cf.mcParallelSimul(cf.European(0.0, 0.5), mdl, num=num).payoffs == 1.0)
