"""FP64 Dupire paths where the grouped checkpoints, the narrow and the wide
smoothing zone and the layouts can go wrong, against the CPU oracle: step
counts around a multiple of four (the last up to three checkpoints lie in
rows), zones under and over the width of the narrow form and one that reaches
down to 0, the FULL and the LEAN layout, both sources of normals.  Payoffs to
1e-11, risks to 1e-10 of their scale, the bounds of the parity tests."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("weeks", [1, 3, 4, 5, 66])
@pytest.mark.parametrize("smooth", [0.05, 0.3, 1.7])
@pytest.mark.parametrize("n_spots", [30, 260])
def test_barrier_paths_and_risks(engine, weeks, smooth, n_spots):
    # the barrier near the spot, so that short paths meet the zone
    mk = W.dupire_args(n_spots)
    pk = W.barrier_args(strike=95.0, barrier=108.0 if weeks < 60 else 150.0, maturity=weeks / 52.0, smooth=smooth)
    mdl, prd, om, op = cf.Dupire(**mk), cf.UOC(**pk), po.Model(**mk), po.Product(**pk)
    n = 700
    res = cf.mcParallelSimulAAD(prd, mdl, n, weights=[1.0, 0.4], per_path=True)
    pay, _, risks = po.aad(om, op, n, weights=[1.0, 0.4])
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()
    price = cf.mcParallelSimul(prd, mdl, n)
    np.testing.assert_allclose(price.payoffs, pay, rtol=1e-11, atol=1e-11)


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("weeks", [5, 67])
def test_mrg_barrier_paths_and_risks(engine, mode, weeks):
    mk = W.dupire_args(30)
    pk = W.barrier_args(strike=95.0, barrier=120.0, maturity=weeks / 52.0)
    mdl, prd, om, op = cf.Dupire(**mk), cf.UOC(**pk), po.Model(**mk), po.Product(**pk)
    num = cf.NumericalParam(numPath=500, useSobol=False, aadMode=mode)
    res = cf.mcParallelSimulAAD(prd, mdl, num=num, per_path=True)
    pay, _, risks = po.aad(om, op, 500, 0, mrg=(num.seed1, num.seed2))
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("smooth,barrier", [(0.03125, 0.96875), (0.125, 0.875)])
@pytest.mark.parametrize("again", [False, True])
def test_exactly_zero_factor(engine, again, smooth, barrier, mode):
    """Spot 1, whose logarithm and exponential are exact, on barrier + width at
    the first date, in the narrow and the wide form of the zone; without vol on
    every date (more than one zero factor)."""
    assert barrier + smooth == 1.0
    vol = 0.0 if again else 0.2
    mk = dict(spot=1.0, spots=[0.5, 1.0, 2.0], times=[0.5, 1.0], vols=[[vol, vol]] * 3, maxDt=1.0 / 52.0)
    pk = W.barrier_args(strike=0.75, barrier=barrier, maturity=0.25, freq=1.0 / 12.0, smooth=smooth)
    w = [1e9, 0.4]
    res = cf.mcParallelSimulAAD(cf.UOC(**pk), cf.Dupire(**mk), weights=w, per_path=True,
                                num=cf.NumericalParam(numPath=500, aadMode=mode))
    pay, _, risks = po.aad(po.Model(**mk), po.Product(**pk), 500, weights=w)
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11)
    assert np.all(res.payoffs[:, 0] == 0.0)
    assert again or np.abs(risks[0]) > 1e6         # (the oracle: the zero factor carries the delta)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()
