"""Black-Scholes barrier paths, whose samples are worked only where a path is in
the smoothing zone: payoffs and risks against the CPU oracle for step counts
around a multiple of four, zones that most, some and none of the paths meet
(one that reaches down to 0), calls and puts with and without weight on the
vanilla, both measures, both adjoint variants and both sources of normals.
FP64: payoffs to 1e-11, risks to 1e-10 of their scale, the bounds of the parity
tests."""
import numpy as np
import pytest

import compfinance_amd as cf
import pyoracle as po
from compfinance_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [cf.AAD_CHECKPOINT, cf.AAD_RECOMPUTE])
@pytest.mark.parametrize("sobol,put", [(True, False), (False, True)])
@pytest.mark.parametrize("spot_measure", [False, True])
@pytest.mark.parametrize("weights", [[1.0, 0.0], [0.7, 0.4]])
@pytest.mark.parametrize("weeks", [1, 3, 4, 5, 67])
@pytest.mark.parametrize("barrier,smooth", [(104.0, 0.02), (118.0, 0.05), (110.0, 1.2), (900.0, 0.05)])
def test_paths_and_risks(engine, barrier, smooth, weeks, weights, spot_measure, sobol, put, mode):
    mk = dict(spot=100.0, vol=0.2, spotMeasure=spot_measure, rate=0.03, div=0.01)
    pk = W.barrier_args(strike=99.0, barrier=barrier, maturity=weeks / 52.0, smooth=smooth, put=put)
    n = 300
    num = cf.NumericalParam(numPath=n, useSobol=sobol, aadMode=mode)
    res = cf.mcParallelSimulAAD(cf.UOC(**pk), cf.BlackScholes(**mk), num=num, weights=weights, per_path=True)
    kw = {} if sobol else dict(mrg=(num.seed1, num.seed2))
    pay, _, risks = po.aad(po.Model(**mk), po.Product(**pk), n, weights=weights, **kw)
    np.testing.assert_allclose(res.payoffs, pay, rtol=1e-11, atol=1e-11)
    assert np.abs(res.risks - risks).max() <= 1e-10 * np.abs(risks).max()
