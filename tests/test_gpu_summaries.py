"""Edges of the cross-path and along-time reductions: chunk remainders, more
chunks than a wave has lanes, histogram chunks between their bounds, and the
load groups of the along-axis kernel below and above one block per CU."""
import numpy as np
import pytest

from sdepy_amd import _lib

torch = pytest.importorskip('torch')
pytestmark = pytest.mark.gpu


def _sample(rows, n, dtype):
    x = np.random.default_rng(rows * 7 + n).standard_normal((rows, n)).astype(dtype)
    return x, torch.from_numpy(x).cuda()


def _code(dtype):
    return _lib.F32 if dtype == np.float32 else _lib.F64


@pytest.mark.parametrize('dtype', [np.float32, np.float64])
@pytest.mark.parametrize('rows,n', [(1, 1), (5, 16384), (3, 16385), (2, 65 * 16384 + 3),
                                    (67, 4099)])
def test_row_reductions(rows, n, dtype):
    lib, x, code = _lib.lib(), *_sample(rows, n, dtype)[1:], _code(dtype)
    host = x.cpu().numpy().astype(np.float64)
    nws = max(lib.sdegpu_moments_workspace(rows, n), lib.sdegpu_mc_workspace(rows, n))
    ws = torch.empty(nws, dtype=torch.uint8, device='cuda')
    f64 = dict(dtype=torch.float64, device='cuda')
    mean, m2, mm, sums = (torch.empty(s, **f64) for s in (rows, rows, (rows, 3), (rows, 5)))
    centre = torch.zeros(rows, **f64)
    _lib.check(lib.sdegpu_path_moments(_lib.ptr(x), code, rows, n, _lib.ptr(mean),
                                       _lib.ptr(m2), _lib.ptr(ws), nws, _lib.stream()))
    _lib.check(lib.sdegpu_mc_minmax(_lib.ptr(x), code, rows, n, 0, _lib.ptr(mm), _lib.ptr(ws),
                                    nws, _lib.stream()))
    _lib.check(lib.sdegpu_mc_moments(_lib.ptr(x), code, rows, n, 0, _lib.ptr(centre),
                                     _lib.ptr(sums), _lib.ptr(ws), nws, _lib.stream()))
    # sums of n FP64 terms in any order: n 2^-53 of the terms' absolute sum
    tol = 2 * n * 2.0 ** -53
    d = host - host.mean(axis=1, keepdims=True)
    scale = np.abs(host).sum(axis=1) + 1
    assert (np.abs(mean.cpu().numpy() - host.mean(axis=1)) <= tol * scale).all()
    assert (np.abs(m2.cpu().numpy() - (d * d).sum(axis=1))
            <= 8 * tol * ((host - host[:, :1]) ** 2).sum(axis=1) + 1e-300).all()
    assert (mm.cpu().numpy() == np.stack(
        [host.min(axis=1), host.max(axis=1), np.zeros(rows)], axis=1)).all()
    want = np.stack([(host ** k).sum(axis=1) for k in (1, 2, 3, 4, 1)], axis=1)
    size = np.stack([(np.abs(host) ** k).sum(axis=1) for k in (1, 2, 3, 4, 1)], axis=1)
    assert (np.abs(sums.cpu().numpy() - want) <= 2 * tol * size + 1e-300).all()


@pytest.mark.parametrize('rows,n,bins', [(1, 4096, 7), (1, 4097, 100), (3, 8191, 4096),
                                         (1, 500_000, 100), (40, 500_001, 33), (2, 9001, 5000)])
def test_histogram_chunks(rows, n, bins):
    lib, (host, x) = _lib.lib(), _sample(rows, n, np.float32)
    edges = np.linspace(-3, 3, bins + 1)
    ed = torch.from_numpy(np.tile(edges, (rows, 1))).cuda()
    counts = torch.empty((rows, bins + 1), dtype=torch.int64, device='cuda')
    _lib.check(lib.sdegpu_mc_histogram(_lib.ptr(x), _lib.F32, rows, n, 0, _lib.ptr(ed), bins, 0,
                                       _lib.ptr(counts), _lib.stream()))
    got = counts.cpu().numpy()
    for r in range(rows):
        want = np.histogram(host[r].astype(np.float64), bins=edges)[0]
        assert (got[r, :bins] == want).all() and got[r, bins] == n - want.sum()


@pytest.mark.parametrize('dtype', [np.float32, np.float64])
@pytest.mark.parametrize('n', [1, 2, 4, 5, 8, 9, 12, 21])
@pytest.mark.parametrize('cols', [1023, 1024, 300_001, 300_000])
def test_along_axis_groups(n, cols, dtype):
    lib, (host, x) = _lib.lib(), _sample(n, cols, dtype)
    code = _code(dtype)
    for op, ref in ((_lib.REDUCE_MIN, host.min(axis=0)), (_lib.REDUCE_MAX, host.max(axis=0)),
                    (_lib.REDUCE_SUM, host.sum(axis=0)), (_lib.REDUCE_MEAN, host.mean(axis=0)),
                    (_lib.REDUCE_VAR, host.var(axis=0)), (_lib.REDUCE_STD, host.std(axis=0))):
        out = torch.empty(cols, dtype=x.dtype, device='cuda')
        _lib.check(lib.sdegpu_axis_reduce(_lib.ptr(x), code, 1, n, cols, 0, cols, None, op, code,
                                          0, _lib.ptr(out), _lib.stream()))
        assert np.array_equal(out.cpu().numpy(), ref)


@pytest.mark.parametrize('rows,n', [(1, 4096), (60, 40_001), (253, 9000)])
@pytest.mark.parametrize('bins', [1024, 1025, 3000, 4096, 4097])
def test_histogram_chunks_of_many_bins(rows, n, bins):
    """Bin counts around the bounds at which the number of blocks changes."""
    test_histogram_chunks(rows, n, bins)
