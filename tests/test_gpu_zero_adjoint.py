"""Paths whose adjoint is zero (the vanilla out of the money, a breach without
weight on the vanilla) are left out of the reverse sweep: risks against the
CPU oracle's tape where all paths are such, none, and some, with and without
weight on the vanilla, calls and puts, both layouts, both adjoint variants and
both sources of normals.  FP64 to 1e-10 of the risks' scale (the bound of the
parity tests); zero risks are exactly zero."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(mk, product, oracle, weights, mode, sobol):
    n = 700
    num = cf.NumericalParam(numPath=n, useSobol=sobol, aadMode=mode)
    res = cf.mcParallelSimulAAD(product, cf.Dupire(**mk), num=num, weights=weights)
    kw = {} if sobol else dict(mrg=(num.seed1, num.seed2))
    _, _, risks = po.aad(po.Model(**mk), oracle, n, weights=weights, **kw)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("sobol,put", [(True, False), (False, True)])
@pytest.mark.parametrize("weights", [[1.0, 0.0], [1.0, 0.4], [0.0, 1.0]])
@pytest.mark.parametrize("strike", [1.0, 105.0, 1.0e4])
@pytest.mark.parametrize("weeks,n_spots", [(7, 30), (66, 30), (66, 260)])
def test_barrier(engine, weeks, n_spots, strike, weights, sobol, put, mode):
    mk = W.dupire_args(n_spots)
    pk = W.barrier_args(strike=strike, barrier=112.0, maturity=weeks / 52.0, put=put)
    check(mk, cf.UOC(**pk), po.Product(**pk), weights, mode, sobol)


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("strike", [1.0, 100.0, 1.0e4])
def test_european(engine, strike, mode):
    mk, pk = W.dupire_args(30), dict(strike=strike, exerciseDate=1.0)
    check(mk, cf.European(**pk), po.Product(**pk), [1.0], mode, True)


@pytest.mark.parametrize("strike,weights", [(120.0, [1.0, 0.0]), (100.0, [1.0, 0.3]), (1.0, [0.0, 1.0]),
                                            (1.0e4, [1.0, 0.0]), (118.0, None)])
@pytest.mark.parametrize("n,first", [((1 << 19) + 77, 0), (1 << 20, 1000)])
def test_paths_of_several_blocks_are_swept_together(engine, n, first, strike, weights):
    """A wave with several blocks of 64 paths gathers the swept ones: the call
    equals the path-weighted mean of calls small enough for one block a wave.
    The same terms in another order, to 1e-11 of their scale."""
    mdl = cf.Dupire(**W.dupire_args(30))
    prd = cf.European(strike, 0.75) if weights is None else cf.UOC(**W.barrier_args(strike=strike, maturity=0.75))
    weights = weights or [1.0]
    res = cf.mcParallelSimulAAD(prd, mdl, num=cf.NumericalParam(numPath=n, firstPath=first), weights=weights)
    part, total = 1 << 17, 0.0
    for lo in range(0, n, part):
        m = min(part, n - lo)
        total = total + m * cf.mcParallelSimulAAD(
            prd, mdl, num=cf.NumericalParam(numPath=m, firstPath=first + lo), weights=weights).risks
    assert np.abs(res.risks - total / n).max() <= 1e-11 * np.abs(total / n).max()


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("precision", [cf.FP64, cf.FP32])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("model", ["dupire", "bs"])
def test_weights_out_of_range_show(engine, model, bad, precision, mode):
    """A weight that is not finite makes the risks NaN on a path out of the money
    too (0 times it), so no path is left out: risks of a strike no path reaches."""
    mdl = cf.Dupire(**W.dupire_args(30)) if model == "dupire" else cf.BlackScholes(100.0, 0.2, False, 0.01, 0.0)
    prd = cf.UOC(**W.barrier_args(strike=1.0e4, maturity=0.2))
    num = cf.NumericalParam(numPath=200, precision=precision, aadMode=mode)
    for weights in ([1.0, bad], [bad, 0.5]):
        assert np.isnan(cf.mcParallelSimulAAD(prd, mdl, weights=weights, num=num).risks[0])
    assert np.all(cf.mcParallelSimulAAD(prd, mdl, weights=[1.0, 0.5], num=num).risks == 0.0)


@pytest.mark.parametrize("weeks,barrier", [(0, False)] + [(n, b) for n in (1, 3, 4, 5) for b in (False, True)])
def test_short_timelines_of_several_blocks(engine, weeks, barrier):
    """Gathered sweeps of no step, of steps in rows alone, and of one group of
    four: as the calls of one block a wave, to 1e-11 of their scale."""
    mdl = cf.Dupire(**W.dupire_args(30))
    prd = cf.UOC(**W.barrier_args(strike=98.0, barrier=107.0, maturity=weeks / 52.0)) if barrier else \
        cf.European(98.0, weeks / 52.0)
    n, part, total = (1 << 19) + 77, 1 << 17, 0.0
    res = cf.mcParallelSimulAAD(prd, mdl, num=cf.NumericalParam(numPath=n))
    for lo in range(0, n, part):
        m = min(part, n - lo)
        total = total + m * cf.mcParallelSimulAAD(prd, mdl, num=cf.NumericalParam(numPath=m, firstPath=lo)).risks
    assert np.abs(res.risks - total / n).max() <= 1e-11 * np.abs(total / n).max()
    if weeks == 0:
        assert abs(res.risks[0] - 1.0) < 1e-12 and np.all(res.risks[1:] == 0.0)
