"""Itemized risk of Europeans on Dupire, where the calls of a maturity share
their sweeps: column k equals the single AAD run with one-hot weights on payoff
k, on the same paths, to the rounding of the adjoint sums (1e-12 of the
largest risk in FP64; FP32 takes the same FP32 steps, so the same), at list
lengths around a wave and a block, with and without the merged last block of
Sobol indices, with equal strikes, strikes no path and every path passes, a
call of today, step counts around a multiple of four, both places of the
local-vol table, and mrg32k3a paths; and the oracle's tape on one case."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu

SURFACE = dict(maturities=[0.25, 1.0, 1.0, 1.0, 1.0, 0.5, 0.5, 0.02], strikes=[100.0, 120.0, 80.0, 1.0, 80.0, 95.0, 900.0, 101.0])


def _one_hot(prd, mdl, num):
    means, risks = cf.mcParallelSimulAADMulti(prd, mdl, num=num)
    npay = len(prd.payoffLabels())
    assert risks.shape == (mdl.numParams(), npay)
    for k in range(npay):
        one = cf.mcParallelSimulAAD(prd, mdl, weights=np.eye(npay)[k], num=num)
        np.testing.assert_array_equal(means, one.payoff_means)
        tol = 1e-12 * max(np.abs(one.risks).max(), 1e-300)
        assert np.abs(risks[:, k] - one.risks).max() <= tol, (k, np.abs(risks[:, k] - one.risks).max())
    return means, risks


@pytest.mark.parametrize("prec", [cf.FP64, cf.FP32])
@pytest.mark.parametrize("paths,first", [(1, 0), (64, 0), (65, 3), (1024, 0), (4097, 1061), (70001, 0)])
def test_columns_are_the_one_hot_runs(engine, prec, paths, first):
    mdl, prd = cf.Dupire(**W.dupire_args(30)), cf.Europeans(**SURFACE)
    _one_hot(prd, mdl, cf.NumericalParam(numPath=paths, firstPath=first, precision=prec))


@pytest.mark.parametrize("prec", [cf.FP64, cf.FP32])
@pytest.mark.parametrize("n_spots,maturity", [(60, 4.0), (60, 2.98), (1, 0.5), (200, 0.6)])
@pytest.mark.parametrize("sobol", [True, False])
def test_grids_and_generators(engine, prec, n_spots, maturity, sobol):
    args = W.dupire_args(max(n_spots, 2))
    if n_spots == 1:
        args.update(spots=args["spots"][:1], vols=np.asarray(args["vols"])[:1])
    mdl = cf.Dupire(**args)
    prd = cf.Europeans(maturities=[maturity, maturity, maturity / 2], strikes=[90.0, 110.0, 100.0])
    _one_hot(prd, mdl, cf.NumericalParam(numPath=2500, precision=prec, useSobol=sobol))


def test_today_and_zero_vols(engine):
    """A call exercised today (no steps), and local vols of 0, which the
    shared sweeps leave to the sweep per payoff."""
    mdl = cf.Dupire(**W.dupire_args(30))
    _one_hot(cf.Europeans(maturities=[0.0, 0.5], strikes=[90.0, 100.0]), mdl, cf.NumericalParam(numPath=500))
    args = W.dupire_args(30)
    vols = np.array(args["vols"])
    vols[:5] = 0.0
    _one_hot(cf.Europeans(maturities=[0.5, 0.5], strikes=[90.0, 100.0]), cf.Dupire(**dict(args, vols=vols)),
             cf.NumericalParam(numPath=500))


def test_columns_match_the_oracle_tape(engine):
    mk = W.dupire_args(30)
    mdl, prd, om, op = cf.Dupire(**mk), cf.Europeans(**SURFACE), po.Model(**mk), po.Product(**SURFACE)
    n = 600
    means, risks = cf.mcParallelSimulAADMulti(prd, mdl, num=cf.NumericalParam(numPath=n))
    for k in range(risks.shape[1]):
        _, _, ref = po.aad(om, op, n, k)
        assert np.abs(risks[:, k] - ref).max() <= 1e-10 * max(np.abs(ref).max(), 1e-300)


@pytest.mark.parametrize("prec,paths", [(cf.FP64, 260001), (cf.FP32, 450001)])
@pytest.mark.parametrize("calls", [3, 4])
def test_both_sides_of_the_rule_for_few_calls(engine, calls, prec, paths):
    """More buffers than the shared sweeps keep: three calls are swept by the
    payoff, four share."""
    prd = cf.Europeans(maturities=[3.0, 3.0, 1.5, 3.0][:calls], strikes=[90.0, 110.0, 100.0, 95.0][:calls])
    _one_hot(prd, cf.Dupire(**W.dupire_args(30)), cf.NumericalParam(numPath=paths, precision=prec))
