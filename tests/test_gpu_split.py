"""Runs of few paths (k_euler_split: several waves share 64 paths) against the
one-wave-per-path kernel on the same draws, across the path counts at which
the share changes, and against the oracle at the edges of its step chunks."""
import numpy as np
import pytest

import sdepy_amd as sa
from oracle import euler as ora
from sdepy_amd import integration

pytestmark = pytest.mark.gpu

ALONE = 65_537      # the fewest paths that k_euler takes

CORR3 = np.array([[1., .3, -.2], [.3, 1., .1], [-.2, .1, 1.]])
CONFIGS = {
    'wiener2': (sa.wiener_process, dict(vshape=2, mu=.1, sigma=.3, rho=.4)),
    'gbm': (sa.lognorm_process, dict(mu=.05, sigma=.2)),
    'gbm4': (sa.lognorm_process, dict(vshape=4, mu=.05, sigma=.2)),
    'ou': (sa.ornstein_uhlenbeck_process, dict(x0=.3, k=2., theta=.5, sigma=.4)),
    'ou3corr': (sa.ornstein_uhlenbeck_process,
                dict(vshape=3, k=2., theta=.5, sigma=.4, corr=CORR3)),
    'hw2f': (sa.hull_white_process, dict(factors=2, k=np.array([[.1], [.3]]),
                                         sigma=np.array([[.01], [.02]]), rho=.3)),
    'cir': (sa.cox_ingersoll_ross_process, dict(x0=.05, theta=.04, k=2., xi=.2)),
    'heston': (sa.full_heston_process, dict(x0=100., mu=.02, y0=.04, theta=.05, k=2., xi=.3,
                                            rho=-.6)),
    'heston2': (sa.heston_process, dict(vshape=2, x0=100., y0=.04, theta=.05, k=2., xi=.2,
                                        rho=np.array([-.6, .2]))),
    'merton2': (sa.merton_jumpdiff_process, dict(vshape=2, mu=.03, sigma=.2, lam=3., a=-.05,
                                                 b=.1)),
    'kou': (sa.kou_jumpdiff_process, dict(mu=.03, sigma=.2, lam=3., a=.1, b=.05, pa=.4)),
}


def _run(name, dtype, paths, tt, steps, **more):
    cls, kw = CONFIGS[name]
    info = {}
    x = cls(paths=paths, dtype=dtype, steps=steps, info=info, rng=np.random.default_rng(3),
            **kw, **more)(tt)
    return (x if isinstance(x, tuple) else (x,)), info


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('name', sorted(CONFIGS))
def test_split_equals_one_wave_per_path(gpu, name, dtype):
    tt = np.linspace(0., 1., 8)
    ref, ref_info = _run(name, dtype, ALONE, tt, 43)
    # FP64: the parity bar; FP32: the bar of the FP32 sweep, of the values' size
    for paths in (1, 65, 16_384, 16_385, 32_769, ALONE - 1):
        got, info = _run(name, dtype, paths, tt, 43)
        for g, r in zip(got, ref):
            r = r[..., :paths]
            if dtype == np.float64:
                assert np.max(np.abs(g - r) / np.maximum(np.abs(r), 1e-3)) < 1e-12, paths
            else:
                assert np.max(np.abs(g - r)) < 2e-5 * np.max(np.abs(r)), paths
        for key in ('negative_y_count', 'jump_count'):
            if key in info and dtype == np.float64:
                assert np.array_equal(info[key], ref_info[key][..., :paths]), paths
        if 'jump_rate' in info:
            total = info['jump_rate'][:-1] * np.diff(tt) * paths
            assert np.isclose(total.sum(), info['jump_count'].sum(), rtol=1e-12)


@pytest.mark.parametrize('name', ['gbm', 'kou'])
def test_split_antithetic_and_backward(gpu, name):
    """Antithetic halves, and a backward and a forward pass (i0 = 2)."""
    tt = np.linspace(0., 1., 6)
    anti = dict(dw=sa.odd_wiener_source)
    if name == 'kou':
        anti['dj'] = sa.even_cpoisson_source
    for more in (anti, dict(i0=2)):
        ref, _ = _run(name, np.float64, ALONE + 1, tt, 31, **more)
        got, _ = _run(name, np.float64, 1000, tt, 31, **more)
        half = 500 if 'dw' in more else 1000
        assert np.allclose(got[0][..., :half], ref[0][..., :half], rtol=1e-12, atol=0.)
        if 'dw' in more:
            # the trailing halves read the leading ones' draws
            at = (ALONE + 1) // 2
            assert np.allclose(got[0][..., half:], ref[0][..., at:at + half], rtol=1e-12, atol=0.)


@pytest.mark.parametrize('nsteps', [1, 3, 4, 5, 31, 32, 33, 63, 65])
@pytest.mark.parametrize('rows', ['all', 'ends', 'some'])
def test_chunk_edges_match_oracle(gpu, nsteps, rows):
    """Step counts around a chunk (32 steps at one component, 16 at 3), every
    step stored, the last one only, and uneven rows."""
    grid = np.linspace(0., 1., nsteps + 1)
    tt = {'all': grid, 'ends': grid[[0, -1]],
          'some': grid[np.unique(np.r_[0, nsteps // 3, nsteps // 2, nsteps])]}[rows]
    P = 100
    p = sa.lognorm_process(paths=P, steps=grid, mu=.05, sigma=.2, rng=np.random.default_rng(4))
    ref = ora.integrate('lognorm', tt, paths=P, steps=grid,
                        sources={'dw': ora.PhiloxWiener(p.sources['dw'].key, 0, P, ())},
                        x0=1., mu=.05, sigma=.2)
    assert np.max(np.abs(p(tt) / ref - 1)) < 1e-12
    p = sa.ornstein_uhlenbeck_process(paths=P, vshape=3, steps=grid, k=2., theta=.5, sigma=.4,
                                      corr=CORR3, rng=np.random.default_rng(4))
    src = ora.PhiloxWiener(p.sources['dw'].key, 0, P, (3,), corr=CORR3)
    ref = ora.integrate('ou', tt, paths=P, vshape=(3,), steps=grid,
                        sources={'dw': src}, x0=0., k=2., theta=.5, sigma=.4)
    assert np.max(np.abs(p(tt) - ref)) < 1e-12


@pytest.mark.parametrize('paths', [1, 300, 5000])
def test_moments_of_few_paths_fused_and_separate(gpu, monkeypatch, paths):
    """prepare(moments=True) reduces few paths in a pass of its own; the
    kernels with the moments fused in give the same (their partial blocks)."""
    tt = np.linspace(0., 1., 23)

    def moments():
        r = sa.ornstein_uhlenbeck_process(paths=paths, vshape=3, k=2., theta=.5, sigma=.4,
                                          corr=CORR3, rng=np.random.default_rng(5)).prepare(
                                              tt, moments=True)
        r.launch()
        return r._row_mom is not None, r.pmean(), r.pvar(), r.result()
    fused, m, v, x = moments()
    assert not fused
    monkeypatch.setattr(integration, '_SEPARATE_PATHS', 0)
    fused, fm, fv, fx = moments()
    assert fused
    assert np.allclose(x, fx, rtol=0., atol=1e-12)
    for a, b, ref in ((m, fm, x.mean(axis=-1, keepdims=True)),
                      (v, fv, x.var(axis=-1, keepdims=True))):
        assert np.allclose(a, ref, rtol=1e-12, atol=1e-14)
        assert np.allclose(b, ref, rtol=1e-12, atol=1e-14)


@pytest.mark.parametrize('paths', [49_152, 49_153])
def test_three_fp64_cir_components(gpu, paths):
    """On either side of the blocks that three per CU hold at once."""
    tt, kw = np.array([0., .5, 1.]), dict(x0=.05, theta=.04, k=2., xi=.2)
    p = sa.cox_ingersoll_ross_process(paths=paths, vshape=3, corr=CORR3, steps=17,
                                      rng=np.random.default_rng(8), **kw)
    src = ora.PhiloxWiener(p.sources['dw'].key, 0, 100, (3,), corr=CORR3)
    ref = ora.integrate('cir', tt, paths=100, vshape=(3,), steps=17, sources={'dw': src}, **kw)
    assert np.max(np.abs(p(tt)[..., :100] - ref)) < 1e-12
