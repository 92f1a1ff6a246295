"""FP32 jump models on either side of the step counts from which zero counts are decided by
the pass's bound, where jumps are summed in place and where they are deferred, with antithetic halves and with fused
row moments too; counts and values against the oracle, jump by jump."""
import numpy as np
import pytest

import sdepy_amd as sa
from oracle import euler as ora

pytestmark = pytest.mark.gpu

PATHS = 65_602


@pytest.mark.parametrize('how', ['plain', 'antithetic', 'moments'])
@pytest.mark.parametrize('nvar,nsteps', [(1, 12), (1, 95), (1, 96), (2, 159), (2, 160),
                                         (3, 157), (3, 163)])
@pytest.mark.parametrize('lam', [.5, 40.])
def test_forms_match_oracle(gpu, how, nvar, nsteps, lam):
    grid = np.linspace(0., 1., nsteps + 1)
    tt = np.unique(np.r_[grid[::5], grid[-1]])      # too many rows to defer jumps
    _check(how, nvar, grid, tt, lam, 0)


@pytest.mark.parametrize('how', ['plain', 'antithetic', 'moments'])
@pytest.mark.parametrize('nvar,nsteps', [(1, 8), (1, 23), (1, 24), (2, 22), (2, 24), (3, 39),
                                         (3, 40)])
@pytest.mark.parametrize('lam', [.5, 40.])
def test_deferred_forms_match_oracle(gpu, how, nvar, nsteps, lam):
    _check(how, nvar, np.linspace(0., 1., nsteps + 1), np.array([0., 1.]), lam, 1)


@pytest.mark.parametrize('paths', [65_537, 67_328, 67_584, 67_599])
def test_one_component_in_place_every_block(gpu, paths):
    """Rows on and off the 64-byte lines, of a number of blocks that is a multiple of eight
    and one more; paths of every block."""
    grid = np.linspace(0., 1., 97)
    _check('plain', 1, grid, grid, .5, 0, paths, 127)


def _check(how, nvar, grid, tt, lam, deferred, paths=PATHS, every=2_999):
    vshape = () if nvar == 1 else (nvar,)
    jump = dict(lam=lam, a=-.01, b=.02)
    anti = how == 'antithetic'
    info, ref_info = {}, {}
    p = sa.merton_jumpdiff_process(
        paths=paths, vshape=vshape, steps=grid, dtype=np.float32, info=info, mu=.03, sigma=.2,
        dw=sa.odd_wiener_source if anti else None, rng=np.random.default_rng(9), **jump)
    dw, dj = p.sources['dw'], p.sources['dj']
    run = p.prepare(tt, moments=how == 'moments')
    assert all(q.jump_defer == deferred for ps in run.passes for q in ps.probs)
    assert (run._row_mom is not None) == (how == 'moments')
    x = run.run()
    # of antithetic paths the leading half, whose normals and jumps are a plain run's
    at = np.arange(0, paths // 2 if anti else paths, every)
    key = dw.half.key if anti else dw.key
    ref = ora.integrate(
        'jumpdiff', tt, paths=at.size, vshape=vshape, steps=grid, info=ref_info, x0=1., mu=.03,
        sigma=.2, sources={'dw': ora.PhiloxWiener(key, 0, at.size, vshape, path_index=at),
                           'dj': ora.PhiloxCPoisson(dj.key, 0, at.size, vshape, path_index=at,
                                                    **jump)})
    assert np.array_equal(info['jump_count'][..., at], ref_info['jump_count'])
    # up to 163 steps and some 40 jumps, each rounding a state of about 1 to 24 bits a few times
    assert np.max(np.abs(x[..., at] / ref - 1)) < 2e-4
    if how == 'moments':
        assert np.allclose(run.pmean(dtype=np.float64)[..., 0],
                           np.asarray(x, np.float64).mean(axis=-1), rtol=1e-12, atol=0.)
