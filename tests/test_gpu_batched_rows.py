"""Step counts around the 64 steps whose rows a wave of the batched kernel copies
ahead and around its groups of 4 (one component) and 2 steps (two factors), with and
without correlations, against the presets on their own; one path more than a
wave has."""
import hashlib
import json

import numpy as np
import pytest

import sdepy_amd as sa
from sdepy_amd import batched as B

pytestmark = pytest.mark.gpu

NSTEPS = (1, 2, 3, 5, 63, 64, 65, 66, 128, 131)


def _spec(i, nsteps):
    kw = dict(paths=65, steps=nsteps, dtype=np.float32, rng=np.random.default_rng(40 + i))
    hw = dict(x0=.02, theta=.03, sigma=np.array([[.01], [.02]]), k=np.array([[.3], [.1]]))
    return [lambda: sa.lognorm_process(x0=1., mu=.05, sigma=.3, **kw),
            lambda: sa.wiener_process(x0=.2, mu=.05, sigma=.3, **kw),
            lambda: sa.ornstein_uhlenbeck_process(x0=.5, theta=1., k=2., sigma=.3, **kw),
            lambda: sa.hull_white_process(factors=2, rho=.6, **hw, **kw),
            lambda: sa.hull_white_process(factors=2, rho=None, **hw, **kw)][i]()


@pytest.mark.parametrize('i', range(5))
def test_rows_ahead(gpu, i):
    bt = B.BatchedTerminalMoments([(_spec(i, n), (0., 1.)) for n in NSTEPS], autotune=False,
                                  graph=False)
    mean, var = bt.run()
    for j, n in enumerate(NSTEPS):
        x = np.asarray(_spec(i, n)((0., 1.)), np.float64)[-1]
        # FP32 states that are rounded in another order (the bars of the batches' test)
        scale = max(abs(x.mean()), x.std(), 1e-3)
        assert abs(mean[j] - x.mean()) < 1e-5 * scale, n
        assert abs(var[j] - x.var()) < 1e-4 * x.var() + 1e-12, n


def test_points_tuned_for_the_previous_kernel_are_not_used(gpu, tmp_path, monkeypatch):
    """A batch does not take up the launch point that the cache holds for the same
    shape under the tag of the kernel before."""
    path = tmp_path / 'tune.json'
    monkeypatch.setenv('SDEPY_AMD_TUNE_CACHE', str(path))

    def batch():
        specs = [(sa.lognorm_process(paths=1000, steps=20, dtype=np.float32,
                                     rng=np.random.default_rng(3)), (0., 1.))]
        return B.BatchedTerminalMoments(specs, autotune=False, graph=False)
    b = batch()
    old = hashlib.sha1(b'v2' + b.nsteps.tobytes() + b.paths.tobytes() +
                       b.nvars.tobytes()).hexdigest()[:16]
    point = {'blocks': b.cu * 12, 'tile_waves': 16, 'order': 'interleave'}
    path.write_text(json.dumps({old: point}))
    assert batch().tile_waves == 1
    path.write_text(json.dumps({b.sig: point}))
    assert batch().tile_waves == 16
