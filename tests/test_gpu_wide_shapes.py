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


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('cls,kw', [
    (sa.lognorm_process, dict(vshape=9, mu=.05, sigma=.2)),
    (sa.hull_white_process, dict(factors=12, k=.2, sigma=.01)),
    (sa.full_heston_process, dict(vshape=5, y0=.04, theta=.05, k=2., xi=.3, rho=np.full(5, -.5))),
    (sa.merton_jumpdiff_process, dict(vshape=10, lam=3., a=-.05, b=.1))])
def test_order_of_blocks_and_rows_of_partial_lines(gpu, dtype, cls, kw):
    """Block counts around the eights that share an L2, rows on and off 64-byte lines:
    every path, and its counts, as in a run of more paths."""
    tt = np.linspace(0., 1., 4)
    m = kw.get('vshape', kw.get('factors'))
    if cls is not sa.full_heston_process:
        kw = dict(kw, corr=.9 * np.eye(m) + .1)

    def run(paths):
        info = {}
        x = cls(paths=paths, dtype=dtype, steps=13, info=info, rng=np.random.default_rng(3),
                **kw)(tt)
        return (x if isinstance(x, tuple) else (x,)), info
    ref, ref_info = run(1600)
    for paths in (1, 63, 448, 511, 512, 513, 529, 1024, 1087):
        got, info = run(paths)
        for g, r in zip(got, ref):
            r = r[..., :paths]
            assert np.max(np.abs(g - r)) <= (1e-12 if dtype == np.float64 else 2e-5) * \
                np.max(np.abs(r))
        for key in ('negative_y_count', 'jump_count'):
            if key in info:
                assert np.array_equal(info[key], ref_info[key][..., :paths])


@pytest.mark.parametrize('m', [48, 49, 64])
def test_jumps_of_many_coupled_components(gpu, m):
    """FP64 jump models of 48 to 64 coupled components (up to 93 KB of LDS)."""
    P, n, tt = 67, 3, np.linspace(0., 1., 3)
    info, ref_info, jump = {}, {}, dict(lam=6., a=-.05, b=.1)
    p = sa.merton_jumpdiff_process(paths=P, vshape=m, steps=n, corr=_corr(m), info=info, x0=1.,
                                   mu=.03, sigma=.2, rng=np.random.default_rng(5), **jump)
    src = {'dw': ora.PhiloxWiener(p.sources['dw'].key, 0, P, (m,), corr=_corr(m)),
           'dj': ora.PhiloxCPoisson(p.sources['dj'].key, 0, P, (m,), **jump)}
    got = p(tt)
    ref = ora.integrate('jumpdiff', tt, paths=P, vshape=(m,), steps=n, sources=src,
                        info=ref_info, x0=1., mu=.03, sigma=.2)
    assert np.array_equal(info['jump_count'], ref_info['jump_count'])
    assert np.max(np.abs(got / ref - 1)) < 1e-12
