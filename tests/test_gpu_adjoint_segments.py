"""The segment-wise Heston adjoint (FP64 variance) around its 4-step
segments: no whole segment, exactly one, one and a remainder of 1, 2, 3 steps."""
import numpy as np
import pytest

from oracle import greeks as og
from sdepy_amd import greeks as G

pytestmark = pytest.mark.gpu

KEY = (0x0badcafe, 0x12345678)
HPRM = dict(x0=100., r=.02, k=2., theta=.04, xi=.5, rho=-.7, y0=.04)


@pytest.mark.parametrize('n', [3, 4, 5, 6, 7, 12])
@pytest.mark.parametrize('payoff', ['call', 'put'])
def test_segments_and_remainders_match_oracle(gpu, n, payoff):
    P = 1500
    pay, g = og.heston_adjoint(KEY, 6, P, n, 1., strike=100., payoff=payoff, **HPRM)
    ref = np.concatenate(([pay.mean()], g.mean(axis=1)))
    kw = dict(paths=P, steps=n, strike=100., key=KEY, epoch=6, payoff=payoff, **HPRM)
    res = G.heston_greeks(dtype=np.float64, **kw)
    got = np.concatenate(([res.price], [res.greeks[k] for k in og.HESTON_NAMES]))
    # the tolerance of the whole-path sweep's FP64 parity test
    assert np.allclose(got, ref, rtol=1e-10, atol=1e-12 * abs(ref).max())
    # FP32 normals and log price with an FP64 variance: the adjoint and the
    # tangent differ by the FP64 rounding of their derivatives alone
    v = [G.heston_greeks(dtype=np.float32, variance_dtype=np.float64, method=m, **kw)
         for m in ('adjoint', 'tangent')]
    a, t = ([r.price] + [r.greeks[k] for k in og.HESTON_NAMES] for r in v)
    assert np.allclose(a, t, rtol=1e-10, atol=1e-12 * abs(ref).max())
