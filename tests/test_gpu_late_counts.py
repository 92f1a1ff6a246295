"""Deferred jump events that keep the Poisson word and are counted at the next
row: intensities per step on either side of the largest that allows it (22.18: above
it no word is below exp(-lam ds) 2^32), more events than are kept, a backward and a
forward pass; counts and values against the oracle, jump by jump."""
import numpy as np
import pytest

import sdepy_amd as sa
from oracle import euler as ora

pytestmark = pytest.mark.gpu

N = 32      # steps, a row every 16


def _by_pass(source):
    class BySource(source):
        passes = 0

        def begin_pass(self, tag):
            super().begin_pass(tag)
            self.epoch = self.passes
            self.passes += 1
    return BySource


@pytest.mark.parametrize('dtype', [np.float64, np.float32])
@pytest.mark.parametrize('lam', [3., 48., 22.1 * N, 22.3 * N])
@pytest.mark.parametrize('i0', [0, 1])
def test_counts_and_values(gpu, dtype, lam, i0):
    paths, tt, grid = 65_600, np.array([0., .5, 1.]), np.linspace(0., 1., N + 1)
    jump, at = dict(lam=lam, a=-.01, b=.02), np.arange(0, 65_600, 2_011)

    def make(info):
        return sa.merton_jumpdiff_process(paths=paths, steps=grid, info=info, i0=i0, dtype=dtype,
                                          x0=1., mu=.03, sigma=.2,
                                          rng=np.random.default_rng(9), **jump)
    run = make({}).prepare(tt)
    assert all(q.jump_defer == 1 for ps in run.passes for q in ps.probs)
    del run
    info, ref_info = {}, {}
    p = make(info)
    kw, kj = p.sources['dw'].key, p.sources['dj'].key
    x = p(tt)
    ref = ora.integrate(
        'jumpdiff', tt, paths=at.size, steps=grid, i0=i0, info=ref_info, x0=1., mu=.03, sigma=.2,
        sources={'dw': _by_pass(ora.PhiloxWiener)(kw, 0, at.size, (), path_index=at),
                 'dj': _by_pass(ora.PhiloxCPoisson)(kj, 0, at.size, (), path_index=at, **jump)})
    assert np.array_equal(info['jump_count'][at], ref_info['jump_count'])
    # FP32: sums of up to 714 sizes, in 24 bits
    assert np.max(np.abs(x[..., at] / ref - 1)) < (1e-12 if dtype == np.float64 else 1e-3)
