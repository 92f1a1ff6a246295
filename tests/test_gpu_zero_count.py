"""Jump counts where the kernels skip the Poisson inversion: words below the
pass's smallest exp(-lam |ds|) 2^32 are counts of 0.  Intensities of 0 (every
word skipped), tiny, large (none skipped) and changing in time (the bound is
that of the largest); counts and totals equal the oracle's exactly."""
import numpy as np
import pytest

import sdepy_amd as sa
from oracle import euler as ora

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('lam', [0., 1e-7, 2., 60., 'timed'])
@pytest.mark.parametrize('rows', [2, 17])
@pytest.mark.parametrize('paths', [70, 140_000])
def test_counts_match_oracle(gpu, lam, rows, paths):
    n = 16
    if lam == 'timed':
        def lam(t):
            return 0. if t < .3 else 20. * t
    tt = np.linspace(0., 1., rows)
    info = {}
    p = sa.merton_jumpdiff_process(paths=paths, steps=n + 1, info=info, x0=1., mu=.03,
                                   sigma=.2, lam=lam, a=-.05, b=.1,
                                   rng=np.random.default_rng(7))
    kw, kj = p.sources['dw'].key, p.sources['dj'].key
    x = p(tt)
    # the oracle draws jump by jump: 70 of the paths, first and last among them
    at = np.unique(np.linspace(0, paths - 1, 70).astype(int))
    dj = ora.PhiloxCPoisson(kj, 0, at.size, (), lam=lam, a=-.05, b=.1, path_index=at)
    ref_info = {}
    ref = ora.integrate('jumpdiff', tt, paths=at.size, steps=n + 1, info=ref_info,
                        sources={'dw': ora.PhiloxWiener(kw, 0, at.size, (), path_index=at),
                                 'dj': dj}, x0=1., mu=.03, sigma=.2)
    assert np.array_equal(info['jump_count'][at], ref_info['jump_count'])
    if paths == at.size:
        assert np.allclose(info['jump_rate'], ref_info['jump_rate'], rtol=1e-12)
    # every jump is in one row's total
    rate = info['jump_rate'][:-1] * np.diff(tt) * paths
    assert np.isclose(rate.sum(), info['jump_count'].sum(), rtol=1e-12)
    assert np.max(np.abs(x[..., at] / ref - 1)) < 1e-12
