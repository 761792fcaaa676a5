"""FP64 path states that are not numbers (vols so large that a state overflows):
a NaN stays one through the kernels' exponential.  A path in such a state pays
nothing, as in FP32, calls and puts, alone and in a book; and itemized risk is
not finite where the run per payoff is not."""
import numpy as np
import pytest

import compfinance_amd as cf
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu

WEEK = 1.0 / 52.0


def _dupire(vol):
    return cf.Dupire(spot=100.0, spots=[50.0, 100.0, 200.0], times=[0.5, 1.0], vols=[[vol, vol]] * 3, maxDt=WEEK)


def _products(freq):
    bar = dict(strike=100.0, barrier=1e30, maturity=2 * freq, freq=freq)
    call, put = (cf.UOC(**W.barrier_args(put=p, **bar)) for p in (False, True))
    return [call, put, cf.European(100.0, 2 * freq), cf.Book([put, call, cf.Asian(100.0, 2 * freq, freq, 0.0)])]


@pytest.mark.parametrize("product", range(4))
@pytest.mark.parametrize("precision", [cf.FP64, cf.FP32])
def test_dupire_paths_pay_nothing(engine, precision, product):
    """The first step's variance overflows to a state of -infinity, which has no
    interpolated vol: every later state is a NaN."""
    mdl, prd = _dupire(1e200 if precision == cf.FP64 else 1e25), _products(0.125)[product]
    res = cf.mcParallelSimul(prd, mdl, num=cf.NumericalParam(numPath=500, precision=precision))
    assert np.all(res.payoffs == 0.0)


@pytest.mark.parametrize("product", range(4))
def test_black_scholes_paths_pay_nothing(engine, product):
    """A step's deviation overflows, its drift is -infinity: a NaN on the paths of
    a positive normal, a spot of 0 on the others (a quarter of the paths)."""
    mdl = cf.BlackScholes(100.0, 1e308, False, 0.0, 0.0)
    res = cf.mcParallelSimul(_products(4.0)[product], mdl, num=cf.NumericalParam(numPath=2000))
    pays = {0: [0, 1], 1: [], 2: [0], 3: [2, 3, 4]}[product]        # calls
    assert np.all(res.payoffs[:, pays] == 0.0)
    for k in {1: [0, 1], 3: [0, 1]}.get(product, []):               # puts
        assert set(np.unique(res.payoffs[:, k])) == {0.0, 100.0}
        assert 0.7 < (res.payoffs[:, k] == 0.0).mean() < 0.8


def test_itemized_risk_shows_the_paths(engine):
    mdl = _dupire(1e200)
    prd = cf.Europeans([0.25, 0.25, 0.5], [90.0, 110.0, 100.0])
    num = cf.NumericalParam(numPath=500)
    _, risks = cf.mcParallelSimulAADMulti(prd, mdl, num=num)
    for k in range(3):
        one = cf.mcParallelSimulAAD(prd, mdl, weights=np.eye(3)[k], num=num).risks
        assert not np.all(np.isfinite(one))
        np.testing.assert_array_equal(np.isfinite(risks[:, k]), np.isfinite(one))
