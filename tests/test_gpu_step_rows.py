"""The steps whose constants a wave multiplies out ahead (64 at a time; 16 with
row moments): step counts around those blocks, a last wave with one lane,
constants that change at every step, backward steps, with and without
correlation, against the runs of few paths, which read the table's rows."""
import numpy as np
import pytest

import sdepy_amd as sa
from sdepy_amd import integration

pytestmark = pytest.mark.gpu

ALONE = 65_537      # the fewest paths that one wave steps alone; its last wave has one

CONFIGS = {
    'wiener': (sa.wiener_process, dict(mu=lambda t: .1 + t, sigma=.3)),
    'gbm': (sa.lognorm_process, dict(mu=.05, sigma=lambda t: .2 + .1 * t)),
    'heston': (sa.full_heston_process, dict(x0=100., mu=.02, y0=.04, theta=.05, k=2., xi=.3,
                                            rho=-.6)),
    'heston_uncorrelated': (sa.full_heston_process, dict(
        x0=1., mu=lambda t: .02 * t, sigma=lambda t: 1. + t, y0=.01, k=lambda t: 1. + t,
        theta=lambda t: .04 + .02 * t, xi=lambda t: .5 - .1 * t, rho=0.)),
    'merton': (sa.merton_jumpdiff_process, dict(mu=.03, sigma=.2, lam=3., a=-.05, b=.1)),
}


def _process(name, dtype, paths, nsteps, info):
    cls, kw = CONFIGS[name]
    return cls(paths=paths, dtype=dtype, steps=np.linspace(0., 1., nsteps + 1), info=info,
               rng=np.random.default_rng(11), i0=1 if nsteps > 1 else 0, **kw)


def _stack(x):
    return np.stack(x) if isinstance(x, tuple) else x[None]


def _close(got, ref, dtype):
    # the bars of the few-path runs against the others: FP64 parity; FP32 by size
    if dtype == np.float64:
        return np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 1e-3)) < 1e-12
    return np.max(np.abs(got - ref)) < 2e-5 * np.max(np.abs(ref))


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('nsteps', [1, 2, 15, 16, 17, 63, 64, 65, 131])
@pytest.mark.parametrize('name', sorted(CONFIGS))
def test_rows_equal_table(gpu, monkeypatch, name, nsteps, dtype):
    grid = np.linspace(0., 1., nsteps + 1)
    tt = grid[np.unique([0, nsteps // 3, nsteps // 2, nsteps])]
    few = 70
    ref_info, info = {}, {}
    ref = _stack(_process(name, dtype, few, nsteps, ref_info)(tt))
    got = _stack(_process(name, dtype, ALONE, nsteps, info)(tt))
    assert _close(got[..., :few], ref, dtype)
    assert np.isfinite(got).all()
    for key in ('negative_y_count', 'jump_count'):
        if key in info and dtype == np.float64:
            assert np.array_equal(info[key][..., :few], ref_info[key])
    # the row moments fused in
    monkeypatch.setattr(integration, '_SEPARATE_PATHS', 0)
    run = _process(name, dtype, few, nsteps, {}).prepare(tt, moments=True)
    run.launch()
    assert run._row_mom is not None
    x = run.result()
    assert _close(_stack(x), ref, dtype)
    first = _stack(x)[0].astype(np.float64)
    mean = _stack(run.pmean())[0]
    assert np.allclose(np.squeeze(mean), first.mean(axis=-1), rtol=1e-6, atol=1e-12)


@pytest.mark.parametrize('name', ['gbm', 'heston', 'heston_uncorrelated'])
def test_f32_whole_numbers_as_from_the_table(gpu, name):
    # FP32: the variance (its sign is counted) and lognormal values (histograms
    # bin them) carry the rounding of the table's rows, bit for bit
    nsteps, few = 131, 5000
    tt = np.linspace(0., 1., nsteps + 1)[[0, 40, nsteps]]
    ref_info, info = {}, {}
    ref = _stack(_process(name, np.float32, few, nsteps, ref_info)(tt))[-1]
    got = _stack(_process(name, np.float32, ALONE, nsteps, info)(tt))[-1]
    assert np.array_equal(got[..., :few], ref)
    if 'negative_y_count' in info:
        assert np.array_equal(info['negative_y_count'][..., :few], ref_info['negative_y_count'])
