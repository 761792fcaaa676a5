"""The barriers of a book where their shared update and the reverse's zone
tests can go wrong, against the CPU oracle: one, four, five and sixteen
barriers (the kernels update them by fours), their zones in no order, with one
schedule and with several schedules and maturities (some samples observe a part
of them), and smoothing factors that are exactly zero (the spot on barrier +
width today).  FP64 payoffs
to 1e-11 and risks to 1e-10 of their scale, the bounds of the parity tests;
FP32 prices to 0.1 standard errors of FP64."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu

WEEK = 1.0 / 52.0


def _check(parts, mk, n=900, modes=(cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE)):
    mdl = cf.Dupire(**mk) if "spots" in mk else cf.BlackScholes(**mk)
    om, op = po.Model(**mk), po.Product(parts=[kw for _, kw in parts])
    cls = {"barrier": cf.UOC, "asian": cf.Asian, "europeans": cf.Europeans}
    prd = cf.Book([cls[k](**kw) for k, kw in parts])
    w = np.linspace(1.3, 0.4, len(prd.payoffLabels()))
    pay, _, risks = po.aad(om, op, n, weights=w)
    for mode in modes:
        res = cf.mcParallelSimulAAD(prd, mdl, weights=w, per_path=True, num=cf.NumericalParam(numPath=n, aadMode=mode))
        np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11)
        assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max(), mode
    np.testing.assert_allclose(cf.mcParallelSimul(prd, mdl, n).payoffs, pay, rtol=1e-11, atol=1e-11)
    return mdl, prd


@pytest.mark.parametrize("count", [1, 4, 5, 16])
@pytest.mark.parametrize("mixed", [False, True])
def test_barrier_counts_and_schedules(engine, count, mixed):
    rng = np.random.default_rng(count)
    parts = []
    for i in range(count):
        mat = 1.0 if not mixed else (0.5, 1.0, 0.75)[i % 3]
        freq = WEEK if not mixed or i % 2 == 0 else 1.0 / 4.0
        parts.append(("barrier", W.barrier_args(strike=float(rng.uniform(90, 110)), barrier=float(rng.uniform(112, 150)),
                                                maturity=mat, freq=freq, smooth=float(rng.choice([0.02, 0.05])),
                                                put=bool(mixed and i % 5 == 4))))
    if mixed:
        parts += [("asian", dict(strike=99.0, maturity=1.0, fixingFreq=1 / 12, snapFreq=WEEK)),
                  ("europeans", dict(maturities=[0.5, 1.0], strikes=[95.0, 105.0]))]
    mdl, prd = _check(parts, W.dupire_args(30))
    n = 1 << 16
    r64 = cf.mcParallelSimul(prd, mdl, n, per_path=False, precision=cf.FP64)
    r32 = cf.mcParallelSimul(prd, mdl, n, per_path=False, precision=cf.FP32)
    assert np.all(np.abs(r32.means - r64.means) <= 0.1 * r64.std_errs)


@pytest.mark.parametrize("model", ["dupire", "bs"])
@pytest.mark.parametrize("twice", [False, True])
def test_exactly_zero_factors(engine, model, twice):
    """Spot 1, whose logarithm and exponential are exact, on barrier + width at
    the first date (one zero factor); with a frozen spot on two dates (two)."""
    vol = 0.0 if twice else 0.2
    if model == "dupire":
        mk = dict(spot=1.0, spots=[0.5, 1.0, 2.0], times=[0.5, 1.0], vols=[[vol, vol]] * 3, maxDt=WEEK)
    else:
        mk = dict(spot=1.0, vol=vol, rate=0.0, div=0.0)
    assert 0.875 + 0.125 == 1.0
    zero = W.barrier_args(strike=0.75, barrier=0.875, maturity=0.25, freq=0.25 if twice else 1.0 / 12.0, smooth=0.125)
    other = W.barrier_args(strike=0.8, barrier=1.3, maturity=0.25, freq=1.0 / 12.0, smooth=0.1)
    _check([("barrier", other), ("barrier", zero)], mk)
