"""Books with exactly-zero smoothing factors (the spot on barrier + width) in
FP64, against the CPU oracle, where a mark of the factor kept in the barrier's
state could meet other numbers: weights from 1e-12 to 1e12 of either sign, a
spot of 2^30 in itemized risk, and other factors whose product underflows.
Payoffs to 1e-11 and risks to 1e-10 of their scale, the bounds of the parity
tests."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu

WEEK = 1.0 / 52.0
MODES = [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE]


def _model(kind, scale):
    if kind == "bs":
        return dict(spot=scale, vol=0.2, rate=0.02, div=0.01)
    # spot 1, whose logarithm and exponential are exact
    return dict(spot=1.0, spots=[0.5, 1.0, 2.0], times=[0.5, 1.0], vols=[[0.2, 0.25]] * 3, maxDt=WEEK)


def _parts(scale, last):
    """A barrier on barrier + width today and one that is not."""
    zero = W.barrier_args(strike=0.6 * scale, barrier=0.875 * scale, maturity=0.25, freq=1.0 / 12.0, smooth=0.125)
    other = W.barrier_args(strike=0.8 * scale, barrier=1.3 * scale, maturity=0.5 if last else 0.25, freq=1.0 / 12.0,
                           smooth=0.1)
    assert zero["barrier"] + zero["smooth"] * scale == scale
    return [other, zero]


def _objects(mk, parts):
    mdl = cf.Dupire(**mk) if "spots" in mk else cf.BlackScholes(**mk)
    return mdl, cf.Book([cf.UOC(**k) for k in parts]), po.Model(**mk), po.Product(parts=parts)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("kind", ["bs", "dupire"])
@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("notional", [1e-12, 1.0, -1e6, 1e9, 1e12])
def test_any_weight(engine, notional, last, kind, mode):
    scale = 128.0 if kind == "bs" else 1.0
    mdl, prd, om, op = _objects(_model(kind, scale), _parts(scale, last))
    n, w = 700, notional * np.array([0.7, 0.2, 1.0, 0.4])
    res = cf.mcParallelSimulAAD(prd, mdl, weights=w, per_path=True, num=cf.NumericalParam(numPath=n, aadMode=mode))
    pay, _, risks = po.aad(om, op, n, weights=w)
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11 * scale)
    assert np.all(res.payoffs[:, 2] == 0.0)
    assert np.abs(risks).max() > 0.1 * abs(notional)          # (the zero factor's delta is there)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()


@pytest.mark.parametrize("kind,scale", [("bs", 2.0 ** 30), ("bs", 1.0), ("dupire", 1.0)])
def test_itemized(engine, kind, scale):
    mdl, prd, om, op = _objects(_model(kind, scale), _parts(scale, True))
    n = 700
    _, risks = cf.mcParallelSimulAADMulti(prd, mdl, num=cf.NumericalParam(numPath=n))
    for k in range(4):
        _, _, ref = po.aad(om, op, n, weights=np.eye(4)[k])
        assert np.abs(risks[:, k] - ref).max() <= 1e-10 * np.abs(ref).max(), k


@pytest.mark.parametrize("mode", MODES)
def test_product_of_the_other_factors_underflows(engine, mode):
    """Without vol the forward falls slowly from barrier + width: 260 factors
    under 0.03, of product 0 in double, and a survival factor of exactly 0."""
    mk = dict(spot=128.0, vol=0.0, rate=-1e-3, div=0.0)
    pk = W.barrier_args(strike=64.0, barrier=112.0, maturity=5.0, freq=WEEK, smooth=0.125)
    mdl, prd, om, op = _objects(mk, [pk, dict(pk, barrier=150.0)])
    w = np.array([1.0, 0.2, 0.5, 0.1])
    res = cf.mcParallelSimulAAD(prd, mdl, weights=w, per_path=True, num=cf.NumericalParam(numPath=100, aadMode=mode))
    pay, _, risks = po.aad(om, op, 100, weights=w)
    assert np.all(pay[:, 0] == 0.0) and np.all(res.payoffs[:, 0] == 0.0)
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()
