"""Books of barriers whose smoothing zone has no width in the kernel's precision
(no smoothing in FP32, a width under half an ulp of the barrier in FP64), with
the spot exactly on a barrier today: on such a state nothing happens, above it
the path is breached.  A book's columns are the barrier's own kernel's, in both
precisions, and in FP64 the CPU oracle's (payoffs to 1e-11, risks to 1e-10 of
their scale, the bounds of the parity tests); FP32 to 1e-5 of the spot."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu

W2 = np.array([1.0, 0.3, 0.7, 0.0])


def _case(model, smooth):
    spot = 100.0 if model == "bs" else 1.0
    if model == "bs":
        mk = dict(spot=spot, vol=0.2, rate=0.0, div=0.0)
    else:   # spot 1, whose logarithm and exponential are exact
        mk = dict(spot=spot, spots=[0.5, 1.0, 2.0], times=[0.5, 1.0], vols=[[0.2, 0.25]] * 3, maxDt=1.0 / 52.0)
    mdl = cf.Dupire(**mk) if model == "dupire" else cf.BlackScholes(**mk)
    parts = [W.barrier_args(strike=0.9 * spot, barrier=b * spot, maturity=0.25, freq=1.0 / 12.0, smooth=w)
             for b, w in ((1.0, smooth), (0.98, 0.05))]    # (the other one's zone holds the spot)
    return mk, mdl, parts


@pytest.mark.parametrize("model", ["bs", "dupire"])
@pytest.mark.parametrize("precision,smooth", [(cf.FP32, 0.0), (cf.FP32, 1e-12), (cf.FP32, 0.02), (cf.FP64, 1e-18),
                                              (cf.FP64, 0.0), (cf.FP64, float("nan"))])
def test_columns_are_the_barriers_alone(engine, precision, smooth, model):
    mk, mdl, parts = _case(model, smooth)
    num = cf.NumericalParam(numPath=3000, precision=precision)
    both = cf.mcParallelSimul(cf.Book([cf.UOC(**k) for k in parts]), mdl, num=num).payoffs
    for i, k in enumerate(parts):
        alone = cf.mcParallelSimul(cf.UOC(**k), mdl, num=num).payoffs
        np.testing.assert_allclose(both[:, 2 * i:2 * i + 2], alone, rtol=0, atol=1e-5 * mk["spot"])
    assert both[:, 2].mean() > 0.0


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("model", ["bs", "dupire"])
def test_fp64_is_the_oracle(engine, model, mode):
    mk, mdl, parts = _case(model, 1e-18)
    n = 600
    res = cf.mcParallelSimulAAD(cf.Book([cf.UOC(**k) for k in parts]), mdl, weights=W2, per_path=True,
                                num=cf.NumericalParam(numPath=n, aadMode=mode))
    pay, _, risks = po.aad(po.Model(**mk), po.Product(parts=parts), n, weights=W2)
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11)
    assert pay[:, 0].max() > 0.0
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()
