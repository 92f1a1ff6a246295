"""Coupled blocks at the widths where the wide kernel's shape changes (waves
per 64 paths and components per wave), one component or pair either side,
against the oracle in FP64; path counts with a partial block."""
import numpy as np
import pytest

import sdepy_amd as sa
from oracle import euler as ora

pytestmark = pytest.mark.gpu


def _corr(k):
    g = np.random.default_rng(k)
    a = g.standard_normal((k, k))
    c = a @ a.T + k * np.eye(k)
    return c / np.sqrt(np.outer(np.diag(c), np.diag(c)))


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('m', [9, 12, 13, 16, 17, 21, 22, 24, 25, 32, 33, 48, 49, 64])
def test_lognorm_widths(gpu, m, dtype):
    P, n, tt = 67, 5, np.linspace(0., 1., 3)
    kw = dict(x0=1., mu=.03, sigma=np.linspace(.1, .4, m)[:, None])
    p = sa.lognorm_process(paths=P, vshape=m, dtype=dtype, steps=n, corr=_corr(m),
                           rng=np.random.default_rng(3), **kw)
    src = ora.PhiloxWiener(p.sources['dw'].key, 0, P, (m,), corr=_corr(m))
    ref = ora.integrate('lognorm', tt, paths=P, vshape=(m,), steps=n, sources={'dw': src}, **kw)
    assert np.max(np.abs(p(tt) / ref - 1)) < (1e-12 if dtype == np.float64 else 3e-5)


@pytest.mark.parametrize('n', [5, 6, 7, 8, 9, 12, 13, 16, 17, 24, 25, 32])
def test_heston_widths(gpu, n):
    P, tt = 65, np.linspace(0., 1., 3)
    kw = dict(x0=100., mu=.02, y0=.04, theta=np.linspace(.03, .06, n)[:, None], k=2., xi=.2)
    rho = np.linspace(-.7, .3, n)
    p = sa.full_heston_process(paths=P, vshape=n, steps=5, rho=rho,
                               rng=np.random.default_rng(3), **kw)
    src = ora.PhiloxWiener(p.sources['dw'].key, 0, P, (2 * n,), rho=rho)
    ref = ora.integrate('full_heston', tt, paths=P, vshape=(n,), steps=5, sources={'dw': src},
                        **kw)
    for got, want in zip(p(tt), ref):
        assert np.max(np.abs(got / want - 1)) < 1e-12


@pytest.mark.parametrize('P', [1, 15, 16, 17, 48, 63, 81])
@pytest.mark.parametrize('m', [10, 20, 21, 40])
def test_sixteen_path_groups(gpu, m, P):
    # FP64 steps 16 paths in a wave: groups that are full, partial and without a path
    n, tt = 3, np.linspace(0., 1., 4)
    info, ref_info = {}, {}
    jump = dict(lam=6., a=-.05, b=.1)
    p = sa.merton_jumpdiff_process(paths=P, vshape=m, steps=n, corr=_corr(m), info=info, x0=1.,
                                   mu=.03, sigma=.2, rng=np.random.default_rng(5), **jump)
    src = {'dw': ora.PhiloxWiener(p.sources['dw'].key, 0, P, (m,), corr=_corr(m)),
           'dj': ora.PhiloxCPoisson(p.sources['dj'].key, 0, P, (m,), **jump)}
    got = p(tt)
    ref = ora.integrate('jumpdiff', tt, paths=P, vshape=(m,), steps=n, sources=src,
                        info=ref_info, x0=1., mu=.03, sigma=.2)
    assert np.array_equal(info['jump_count'], ref_info['jump_count'])
    assert np.max(np.abs(got / ref - 1)) < 1e-12
