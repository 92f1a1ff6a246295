"""Host-side logic and the C ABI boundary (CPU tests, no GPU compute).

* libsdegpu.so loads and exports every function include/sdegpu.h declares;
* the ctypes mirrors of the C structs have the C compiler's layout;
* argument validation of the entry points (host code, before any launch)
  returns the documented status codes, mapped to sdepy's exception types;
* timeline consolidation, store-row mapping, parameter tables and argument
  handling of the preset classes agree with the oracle's restatement;
* the process type behaves as sdepy's (construction, ufuncs, indexing,
  host summaries);
* without a GPU every simulation entry point fails loudly.
"""
import ctypes
import os
import re
import subprocess
import sys
import tempfile

import numpy as np
import pytest

import sdepy_amd as sa
from sdepy_amd import _lib, greeks as G
from sdepy_amd import integration as integ
from sdepy_amd.infrastructure import per_component, philox_key, cholesky_packed
from oracle import euler as ora

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, 'include', 'sdegpu.h')


def _declared_functions():
    src = open(HEADER).read()
    src = re.sub(r'/\*.*?\*/', '', src, flags=re.S)
    return sorted(set(re.findall(r'\b(sdegpu_\w+)\s*\(', src)))


def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(_lib.LIB_PATH)
    names = _declared_functions()
    assert len(names) >= 17
    for n in names:
        assert hasattr(lib, n), n
    # and the ctypes bindings give every one of them a prototype
    from sdepy_amd import batched
    bound = _lib.lib()
    G._bind()
    batched._bind()
    for n in names:
        assert getattr(bound, n).argtypes is not None, n


def _c_layout(struct, fields):
    code = '#include <stdio.h>\n#include <stddef.h>\n#include "sdegpu.h"\nint main(){\n'
    code += 'printf("%zu\\n", sizeof({}));\n'.format(struct)
    for f in fields:
        code += 'printf("%zu\\n", offsetof({}, {}));\n'.format(struct, f)
    code += 'return 0;}\n'
    with tempfile.TemporaryDirectory() as td:
        c = os.path.join(td, 'l.c')
        exe = os.path.join(td, 'l')
        open(c, 'w').write(code)
        subprocess.run(['gcc', '-I', os.path.dirname(HEADER), c, '-o', exe], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    return [int(v) for v in out.split()]


@pytest.mark.parametrize('cstruct,pystruct', [
    ('sdegpu_euler_problem', _lib.EulerProblem),
    ('sdegpu_heston_greeks', G.HestonGreeksProblem),
    ('sdegpu_loglin_greeks', G.LogGreeksProblem),
    ('sdegpu_batch_instance', __import__('sdepy_amd.batched', fromlist=['x']).BatchInstance),
    ('sdegpu_batch', __import__('sdepy_amd.batched', fromlist=['x']).Batch),
])
def test_ctypes_layout_matches_c(cstruct, pystruct):
    fields = [f[0] for f in pystruct._fields_]
    got = _c_layout(cstruct, fields)
    assert got[0] == ctypes.sizeof(pystruct)
    for f, off in zip(fields, got[1:]):
        assert getattr(pystruct, f).offset == off, f


def test_philox_host_entry_known_answer():
    c = (ctypes.c_uint32 * 4)(0x243f6a88, 0x85a308d3, 0x13198a2e, 0x03707344)
    k = (ctypes.c_uint32 * 2)(0xa4093822, 0x299f31d0)
    o = (ctypes.c_uint32 * 4)()
    _lib.check(_lib.lib().sdegpu_philox_host(c, k, o))
    assert list(o) == [0xd16cfe09, 0x94fdcceb, 0x5001e420, 0x24126ea1]


def test_entry_point_validation_maps_to_exceptions():
    lib = _lib.lib()
    pr = _lib.EulerProblem()
    pr.model, pr.dtype, pr.nvars, pr.paths = _lib.MODEL_LOGNORM, _lib.F32, 65, 10
    with pytest.raises(NotImplementedError):
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.nvars, pr.nout, pr.ncoef = 1, 1, 1
    with pytest.raises(ValueError):        # table too narrow
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.ncoef, pr.exp_mask = 4, 0           # lognorm must exp its output
    pr.out = 1
    with pytest.raises(ValueError):
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.model, pr.nvars = _lib.MODEL_HESTON, 3
    with pytest.raises(ValueError):        # odd Heston state
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.nvars, pr.nout, pr.ncoef, pr.heston_width = 8, 8, 22, 3
    with pytest.raises(ValueError):        # width 3 does not divide 4 log-x values
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.heston_width, pr.nout = 2, 5
    with pytest.raises(ValueError):        # Heston stores 8 or 4 values
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.nout, pr.exp_mask = 8, 0x0F
    with pytest.raises(ValueError, match='0x33'):   # log x of groups [x x y y]
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.heston_width, pr.exp_mask = 2, 0x33
    pr.comp0, pr.nvars_total = 2, 16
    with pytest.raises(ValueError):        # a group must start on a Heston block
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.comp0 = 12
    with pytest.raises(ValueError):        # components 12..19 outside 16
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.comp0, pr.out0, pr.out_stride = 8, 10, 16
    with pytest.raises(ValueError):        # values 10..17 outside rows of 16
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.out0, pr.info_row_slots = 0, 1025
    with pytest.raises(ValueError, match='info_row_slots'):
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.info_row_slots = -1
    with pytest.raises(ValueError, match='info_row_slots'):
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.info_row_slots = 0
    pr.heston_width = pr.comp0 = pr.nvars_total = pr.out0 = pr.out_stride = 0
    pr.model, pr.nvars, pr.paths = _lib.MODEL_OU, 1, 0
    with pytest.raises(ValueError):
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.paths, pr.nout, pr.ncoef, pr.exp_mask, pr.anti_w = 10, 1, 5, 0, 4
    with pytest.raises(ValueError):        # antithetic half must be paths/2
        _lib.check(lib.sdegpu_euler(pr, None))
    pr.anti_w, pr.anti_j = 5, 5
    with pytest.raises(ValueError):        # antithetic jumps without a jump model
        _lib.check(lib.sdegpu_euler(pr, None))
    with pytest.raises(ValueError):
        _lib.check(lib.sdegpu_path_moments(None, 0, -1, 10, None, None, None, 0, None))
    ax = lib.sdegpu_axis_reduce
    one = ctypes.c_void_p(16)
    with pytest.raises(NotImplementedError):       # unknown dtype
        _lib.check(ax(one, 7, 1, 3, 4, 0, 4, None, _lib.REDUCE_SUM, 0, 0, one, None))
    with pytest.raises(ValueError):                # unknown operation
        _lib.check(ax(one, 0, 1, 3, 4, 0, 4, None, 9, 0, 0, one, None))
    with pytest.raises(NotImplementedError):       # float64 values, float32 sums
        _lib.check(ax(one, 1, 1, 3, 4, 0, 4, None, _lib.REDUCE_MEAN, 0, 0, one, None))
    with pytest.raises(ValueError):                # empty reduced axis
        _lib.check(ax(one, 0, 1, 0, 4, 0, 4, None, _lib.REDUCE_MIN, 0, 0, one, None))
    nine = (ctypes.c_int32 * 9)(*range(9))
    with pytest.raises(NotImplementedError):       # more than 8 listed components
        _lib.check(ax(one, 0, 1, 9, 4, 36, 4, nine, _lib.REDUCE_MAX, 0, 0, one, None))
    with pytest.raises(IndexError):                # negative component
        _lib.check(ax(one, 0, 1, 1, 4, 4, 4, (ctypes.c_int32 * 1)(-1), _lib.REDUCE_MAX,
                      0, 0, one, None))
    assert lib.sdegpu_moments_workspace(3, 70000) == 3 * 5 * 2 * 8   # 16384-path chunks
    with pytest.raises(MemoryError):
        _lib.check(lib.sdegpu_path_moments(ctypes.c_void_p(8), 0, 3, 70000,
                                           ctypes.c_void_p(8), ctypes.c_void_p(8),
                                           ctypes.c_void_p(8), 8, None))


@pytest.mark.parametrize('tt,steps,i0', [
    (np.linspace(0, 1, 11), None, 0), (np.linspace(0, 1, 11), 37, 0),
    ((0., .3, 1.), (.1, .2, .25, .9, 5.), 1), (np.arange(10), 37, 0),
    ((2.,), None, 0), ((0., 1., 2., 3.), 8, -1),
])
def test_timeline_consolidation_matches_oracle(tt, steps, i0):
    a = integ.consolidate_timeline(tt, steps, i0)
    b = ora.consolidate(tt, steps, i0)
    for x, y in zip(a, b):
        assert np.array_equal(x, y) and x.dtype == y.dtype


@pytest.mark.parametrize('bad,exc', [
    (np.ones((2, 3)), ValueError), ((1, 2, 2, 3), ValueError),
    ((3, 2, 1), ValueError)])
def test_timeline_errors(bad, exc):
    with pytest.raises(exc):
        integ.consolidate_timeline(bad, None, 0)
    with pytest.raises(IndexError):
        integ.consolidate_timeline((1., 2.), None, 12)


def test_store_rows_forward_and_backward():
    tt = np.array([0., .3, .5, 1., 1.7, 2.])
    _, _, steps = integ.consolidate_timeline(tt, 23, 3)
    j0 = int(np.nonzero(steps == tt[3])[0][0])
    fwd = integ._store_rows(steps[j0:], tt[3:], lambda j: 3 + j)
    bwd = integ._store_rows(steps[j0::-1], tt[3::-1], lambda j: 3 - j)
    # brute force
    for sp, tp, rows, sgn in ((steps[j0:], tt[3:], fwd, 1), (steps[j0::-1], tt[3::-1], bwd, -1)):
        for s, r in enumerate(rows):
            hit = np.nonzero(tp == sp[s + 1])[0]
            assert r == (3 + sgn * hit[0] if hit.size else -1)
    assert set(fwd[fwd >= 0]) == {4, 5} and set(bwd[bwd >= 0]) == {0, 1, 2}


def test_per_component_and_per_path_rejection():
    assert np.array_equal(per_component(np.array([[1.], [2.]]), (2,), 'k'), [1., 2.])
    assert np.array_equal(per_component(3., (2, 2), 'k'), [3.] * 4)
    with pytest.raises(NotImplementedError):
        per_component(np.arange(5.), (), 'x')       # a value per path


def test_philox_key_reproducible():
    assert philox_key(np.random.default_rng(3)) == philox_key(np.random.default_rng(3))
    assert philox_key(np.random.RandomState(3)) == philox_key(np.random.RandomState(3))
    with pytest.raises(TypeError):
        sa.wiener_source(rng=5)


def test_cholesky_packing_block_diagonal():
    c = np.array([[1, .3, .1], [.3, 1, .2], [.1, .2, 1]])
    L = np.linalg.cholesky(c)
    packed = cholesky_packed(c, (2, 3))
    full = np.zeros((6, 6))
    full[np.tril_indices(6)] = packed
    assert np.allclose(full[:3, :3], L) and np.allclose(full[3:, 3:], L)
    assert np.allclose(full[3:, :3], 0)
    with pytest.raises(ValueError):
        cholesky_packed(c, (2,))


def test_preset_argument_handling_and_tables():
    with pytest.raises(TypeError):
        sa.lognorm_process(paths=3, bogus=1)
    with pytest.raises(ValueError):
        sa.lognorm_process(paths=3, method='rk')
    p = sa.lognorm_process(paths=4, mu=lambda t: .1 * t, sigma=.3)
    rows = p._param_rows(np.array([0., 1., 2.]), np.array([1., 1., 1.]))
    assert np.allclose(rows[:, 0], .1 * np.array([0., 1., 2.]) - .045)
    assert np.allclose(rows[:, 1], .3)
    # OU rows (1 - k ds, k theta ds, sigma); sigma sqrt|ds| folded into L rows
    o = sa.ornstein_uhlenbeck_process(paths=4, vshape=2, theta=np.array([[1.], [2.]]),
                                      k=np.array([[.5], [3.]]), sigma=np.array([[.2], [.4]]),
                                      rho=.3)
    tab, hc = o._coef_table(o.sources['dw'], np.array([0., .25]), np.array([.25, .25]))
    assert hc and tab.shape == (2, 2 + 3 + 6)
    assert np.allclose(tab[0, 5:7], [1 - .125, 1 - .75]) and np.allclose(tab[0, 7:9], [.125, 1.5])
    L = np.linalg.cholesky(np.array([[1, .3], [.3, 1]]))
    assert np.allclose(tab[0, 2:5], [L[0, 0] * .2 * .5, L[1, 0] * .4 * .5, L[1, 1] * .4 * .5])
    h = sa.hull_white_process(paths=4, factors=3, rho=None)
    assert h.wshape == (3,) and h.xshape == ()
    assert h._output_map()[:3] == (1, _lib.OUT_SUM, 3)
    fh = sa.full_heston_process(paths=4, vshape=2, rho=[.1, .2])
    assert fh.wshape == (4,) and fh.sources['dw'].corr.shape == (4, 4)
    st = fh._x0_state(np.float64)
    assert st.shape == (4,) and np.allclose(st, [0, 0, 1, 1])
    he = sa.heston_process(paths=4)
    assert he.xshape == () and he._output_map() == (1, _lib.OUT_FIRST, 1, 1)
    m = sa.merton_jumpdiff_process(paths=4, lam=2., a=-.1, b=.2)
    law, tab = m.sources['dj'].kernel_laws(np.zeros(3), np.full(3, .1))
    assert law == _lib.JUMP_NORMAL and np.allclose(tab, [[-.1, .2, 0.]])
    # Kou, the default uniform y, an exponential and a time-dependent law
    # are drawn in the kernel too; an rvmap'd law is not
    k = sa.kou_jumpdiff_process(paths=4, a=.3, b=.2, pa=.6)
    law, tab = k.sources['dj'].kernel_laws(np.zeros(2), np.full(2, .1))
    assert law == _lib.JUMP_DOUBLE_EXP and np.allclose(tab, [[.3, .2, .6]])
    j = sa.jumpdiff_process(paths=4)
    law, tab = j.sources['dj'].kernel_laws(np.zeros(2), np.full(2, .1))
    assert law == _lib.JUMP_UNIFORM and np.allclose(tab, [[0., 1., 0.]])
    e = sa.jumpdiff_process(paths=4, y=sa.exp_rv(-.25))
    law, tab = e.sources['dj'].kernel_laws(np.zeros(2), np.full(2, .1))
    assert law == _lib.JUMP_DOUBLE_EXP and np.allclose(tab, [[-.25, 1., 1.]])
    td = sa.jumpdiff_process(paths=4, y=sa.norm_rv(a=lambda t: t, b=.1))
    law, tab = td.sources['dj'].kernel_laws(np.array([0., 1.]), np.array([1., 2.]))
    assert law == _lib.JUMP_NORMAL and np.allclose(tab[:, 0, 0], [.5, 2.])
    mapped = sa.jumpdiff_process(paths=4, y=sa.rvmap(np.exp, sa.norm_rv()))
    assert mapped.sources['dj'].kernel_laws(np.zeros(2), np.full(2, .1)) is None
    x0 = sa.ornstein_uhlenbeck_process(paths=3, x0=np.array([1., 2., 3.]))
    assert x0._x0_state(np.float64).shape == (1, 3)     # per-path initial values


def test_process_type_semantics():
    t = np.array([0., 1., 2.])
    x = np.arange(3 * 2 * 5, dtype=float).reshape(3, 2, 5)
    p = sa.process(t, x=x)
    assert p.paths == 5 and p.vshape == (2,) and p.t is not None
    q = np.exp(p)
    assert isinstance(q, sa.process) and np.array_equal(q.t, t)
    r = p + p
    assert isinstance(r, sa.process)
    with pytest.raises(ValueError):
        p + sa.process((0., 5., 6.), x=x)
    s = p.sum()
    assert not isinstance(s, sa.process)
    assert isinstance(p.mean(axis=-1), np.ndarray) and not isinstance(p.mean(axis=-1), sa.process)
    assert p['t', 1].shape == (1, 2, 5) and p['t', 1].t[0] == 1.
    assert p['v', 1].shape == (3, 5)
    assert p['p', 2].shape == (3, 2, 1)
    assert np.array_equal(p[0], x[0])
    c = sa.process(c=[1., 2.])
    assert c.shape == (1, 2, 1)
    v = sa.process(t, v=[1., 2., 3.])
    assert v.shape == (3, 1)
    f = p.interp()
    assert np.allclose(f(.5), (x[0] + x[1]) / 2)
    assert np.allclose(p.rebase((.5, 1.5))[0], (x[0] + x[1]) / 2)
    assert np.allclose(p.tmean()[0], x.mean(axis=0))
    assert np.allclose(p.vmean(), x.mean(axis=1))
    assert np.allclose(p.pmin()[..., 0], x.min(axis=-1))
    assert np.allclose(p.pcopy(), p) and p.pcopy().t is not p.t


@pytest.mark.skipif(_lib.torch_mod().cuda.is_available(), reason='a GPU is present')
def test_no_gpu_fails_loudly():
    with pytest.raises(RuntimeError):
        sa.lognorm_process(paths=3)(np.linspace(0, 1, 3))
    with pytest.raises(RuntimeError):
        sa.process(np.arange(2.), x=np.ones((2, 3))).pmean()
    with pytest.raises(RuntimeError):
        sa.wiener_source(paths=3)(0., 1.)
    with pytest.raises(RuntimeError):
        G.heston_greeks(paths=10, steps=3)


def test_antithetic_sources_host_side():
    """sdepy's _antithetics (infrastructure.py:2047-2098): even path counts
    only, the leading half is an ordinary source, properties delegate."""
    with pytest.raises(ValueError):
        sa.odd_wiener_source(paths=7)
    dw = sa.odd_wiener_source(paths=8, vshape=2, rho=.3,
                              rng=np.random.default_rng(1))
    assert dw.paths == 8 and dw.vshape == (2,) and dw.half.paths == 4
    assert isinstance(dw.half, sa.wiener_source)
    assert not isinstance(dw, sa.wiener_source)
    dj = sa.even_cpoisson_source(paths=6, lam=2., y=sa.norm_rv(0., 1.))
    assert dj.half.kernel_laws(np.zeros(1), np.ones(1)) is not None and dj.paths == 6
    assert sa.odd_dw is sa.odd_wiener_source and sa.even_dj is sa.even_cpoisson_source
    # the oracle's restatement of the wrapper
    from oracle import euler as ora
    src = ora.Antithetic(ora.NumpyWiener(np.random.RandomState(0), 5, ()), -1)
    z = src(0., .5)
    assert z.shape == (10,) and np.array_equal(z[:5], -z[5:])


def test_c_caller_builds_against_the_header():
    """tests/c/abi_smoke.c compiles as C11 with gcc against include/sdegpu.h
    and links libsdegpu.so (run on the GPU by test_gpu_euler)."""
    from sdepy_amd import _build
    exe = _build.build_c_smoke()
    assert exe and os.path.exists(exe)
    out = subprocess.run(['ldd', exe], capture_output=True, text=True).stdout
    assert 'libsdegpu.so' in out


def test_bench_refuses_more_than_one_gpu():
    res = subprocess.run([sys.executable, os.path.join(ROOT, 'bench.py'), '--gpus', '2'],
                         capture_output=True, text=True)
    assert res.returncode == 2 and 'one GPU' in res.stderr


@pytest.mark.parametrize('mode', [None, 'mid', 'forward', 'backward'])
@pytest.mark.parametrize('dtype,paths,vshape,shift', [
    (float, None, (3,), 0), (float, 5, (2, 3), -2), (np.float32, None, (), 0),
    (np.float16, 5, (), 0), (float, None, (2, 3), -4)])
def test_piecewise_semantics(mode, dtype, paths, vshape, shift):
    """piecewise (infrastructure.py:1216-1281): 'nearest' interpolation of
    constant segments centred on, starting at or ending at the given times,
    the earlier segment winning at a shared point; the semantics of the
    reference's test_process.py:776-833."""
    g = np.random.default_rng(7)
    t = np.array((1, 2, 3), dtype=dtype) + shift
    if paths is None:
        v = (1 + g.random((3,) + vshape)).astype(dtype)
        x, kw, npaths = v[..., None], dict(v=v), 1
    else:
        x = (1 + g.random((3,) + vshape + (paths,))).astype(dtype)
        kw, npaths = dict(x=x), paths
    p = sa.piecewise(t, **kw) if mode is None else sa.piecewise(t, mode=mode, **kw)
    assert isinstance(p * p + 2, sa.process)
    assert p.interp_kind == 'nearest'
    assert p.paths == npaths and p.vshape == vshape
    assert p(0).dtype == dtype
    if mode in (None, 'mid'):
        s, idx = (.5, 1, 1.49, 1.51, 2.49, 2.51, 3, 3.5), (0, 0, 0, 1, 1, 2, 2, 2)
    elif mode == 'forward':
        s, idx = (.5, 1, 1.5, 2, 2.01, 2.5, 3, 3.01, 3.5), (0, 0, 0, 0, 1, 1, 1, 2, 2)
    else:
        s, idx = (.5, 1, 1.01, 1.5, 2, 2.01, 2.5, 3, 3.5), (0, 0, 1, 1, 1, 2, 2, 2, 2)
    got = p(np.array(s) + shift)
    assert np.array_equal(got, np.stack([x[i] for i in idx]))
    q = sa.piecewise(t=0., x=x[:1])
    assert np.array_equal(q((-3, 0, 3)), np.stack((x[0], x[0], x[0])))
    with pytest.raises(ValueError):
        sa.piecewise((1, 2), v=(10, 20), mode='zzz')


def test_fd_points_with_zero_parameters():
    """Central-difference sets bump a zero parameter by h itself and divide
    by the difference of the bumped values (no 0/0)."""
    base = dict(x0=100., r=0., k=2., theta=.04, xi=.5, rho=0., y0=.04)
    pts, spans = G.fd_points(base, G.HESTON_GREEKS, 1e-4)
    assert len(pts) == 15 and pts[0] == base
    assert spans['r'] == 2e-4 and spans['rho'] == 2e-4
    assert abs(spans['x0'] - 2e-2) < 1e-13   # 100.01 - 99.99 as rounded
    # a price linear in the parameters: the quotients are its slopes
    slope = dict(x0=.5, r=30., k=-.2, theta=50., xi=-2., rho=.3, y0=40.)

    def price(d):
        return sum(slope[n] * d[n] for n in G.HESTON_GREEKS)
    q = G.fd_quotients([price(d) for d in pts], G.HESTON_GREEKS, spans)
    for n in G.HESTON_GREEKS:
        assert np.isfinite(q[n]) and abs(q[n] - slope[n]) < 1e-8 * max(1., abs(slope[n])), n


def test_batched_takes_float32_processes_only():
    """A default-dtype (float64) process in a batch is refused, not stepped
    in FP32 with other normals."""
    from sdepy_amd import batched
    p = sa.lognorm_process(paths=100, steps=5, x0=1., mu=.05, sigma=.2,
                           rng=np.random.default_rng(1))
    with pytest.raises(NotImplementedError):
        batched._instance(p, (0., 1.))
    p32 = sa.lognorm_process(paths=100, steps=5, x0=1., mu=.05, sigma=.2,
                             dtype=np.float32, rng=np.random.default_rng(1))
    d, tab = batched._instance(p32, (0., 1.))
    assert d.nsteps == 4 and tab.shape[0] == 4


@pytest.mark.parametrize('make,density,support', [
    (lambda: sa.norm_rv(-.1, .15),
     lambda y: np.exp(-(y + .1) ** 2 / (2 * .15 ** 2)) / (.15 * np.sqrt(2 * np.pi)),
     (-3., 3.)),
    (lambda: sa.uniform_rv(-.2, .1), lambda y: np.full_like(y, 1 / .3), (-.2, .1)),
    (lambda: sa.exp_rv(.25), lambda y: np.exp(-y / .25) / .25, (0., 20.)),
    (lambda: sa.exp_rv(-.25), lambda y: np.exp(y / .25) / .25, (-20., 0.)),
    (lambda: sa.double_exp_rv(.2, .3, .6),
     lambda y: np.where(y >= 0, .6 * np.exp(-np.abs(y) / .2) / .2,
                        .4 * np.exp(-np.abs(y) / .3) / .3), (-20., 20.)),
])
def test_jump_law_closed_forms_and_host_draws(make, density, support):
    """mean, var, std and exp_mean of each jump law against quadrature of
    its density, and host draws (rvs) within 4 SE of the mean and var."""
    import scipy.integrate
    law = make()
    lo, hi = support
    pts = [0.] if lo < 0 < hi else None

    def q(f):
        return scipy.integrate.quad(lambda y: f(y) * density(np.array(y)), lo, hi,
                                    points=pts, limit=200)[0]
    m = q(lambda y: y)
    v = q(lambda y: (y - m) ** 2)
    assert abs(q(lambda y: 1.) - 1) < 1e-7
    assert abs(law.mean() - m) < 1e-7 and abs(law.var() - v) < 1e-7
    assert abs(law.std() - np.sqrt(v)) < 1e-7
    assert abs(law.exp_mean() - q(np.exp)) < 1e-6 * q(np.exp)
    y = law.rvs(size=200_000, random_state=np.random.default_rng(3))
    y2 = law.rvs(size=(400, 500), random_state=np.random.RandomState(4))
    assert y2.shape == (400, 500)
    for s in (y, y2.reshape(-1)):
        assert abs(s.mean() - m) < 4 * np.sqrt(v / s.size)
        d2 = (s - m) ** 2
        assert abs(d2.mean() - v) < 4 * d2.std() / np.sqrt(s.size)


def test_jump_law_arguments_and_time_dependence():
    """Domain errors as sdepy's; callable parameters give a law of t; rvmap
    maps the variates (with t first when f takes it)."""
    with pytest.raises(ValueError):
        sa.exp_rv(0.)
    for bad in (dict(a=-1.), dict(b=0.), dict(pa=1.5)):
        with pytest.raises(ValueError):
            sa.double_exp_rv(**bad)
    y = sa.double_exp_rv(a=lambda t: .1 + t, b=.3, pa=.5)
    assert callable(y) and abs(y(1.).mean() - (.5 * 1.1 - .5 * .3)) < 1e-15
    assert sa.exp_rv(2.).exp_mean() == np.inf
    g = np.random.default_rng(0)
    m = sa.rvmap(np.exp, sa.norm_rv(0., 1e-12))
    assert np.allclose(m.rvs(5, random_state=g), 1.)
    mt = sa.rvmap(lambda t, v: t + 0 * v, sa.uniform_rv())
    assert np.allclose(mt(2.5).rvs(4, random_state=g), 2.5)


def test_montecarlo_pdf_and_cdf_from_a_histogram():
    """The kernel estimate spreads each bin's mass as a normal around its
    midpoint: the pdf integrates to 1 and the cdf is its integral; the
    interpolated cdf passes through the cumulated masses at the edges and
    the interpolated pdf through the densities at the midpoints."""
    import scipy.integrate
    import importlib
    M = importlib.import_module('sdepy_amd.montecarlo')
    bins = np.array([-1., -.5, 0., .25, 1., 2.])
    counts = np.array([3., 10., 7., 12., 4.])
    density = counts / counts.sum() / np.diff(bins)
    for bw in (.5, 1., 2.):
        pdf = lambda x: M._histogram_kde(np.asarray(x), density, bins, bw, False)
        cdf = lambda x: M._histogram_kde(np.asarray(x), density, bins, bw, True)
        total = scipy.integrate.quad(pdf, -30, 30, points=list(bins), limit=200)[0]
        assert abs(total - 1) < 1e-8
        for x in (-.7, 0.1, 1.5):
            assert abs(scipy.integrate.quad(pdf, -30, x, limit=200)[0] - cdf(x)) < 1e-8
        assert abs(cdf(1e3) - 1) < 1e-12 and abs(cdf(-1e3)) < 1e-12
    c = M._histogram_interp(bins, density, bins, 'linear', True)
    assert np.allclose(c, np.concatenate(([0.], np.cumsum(counts) / counts.sum())))
    assert M._histogram_interp(np.array([-5., 5.]), density, bins, 'linear', True).tolist() == [0., 1.]
    mid = (bins[:-1] + bins[1:]) / 2
    assert np.allclose(M._histogram_interp(mid, density, bins, 'linear', False), density)
    assert M._histogram_interp(np.array([-5., 5.]), density, bins, 'linear', False).tolist() == [0., 0.]


@pytest.mark.parametrize('dtype,v64', [(_lib.F32, 0), (_lib.F32, 1), (_lib.F64, 0)])
def test_heston_greeks_workspace_serves_both_methods(dtype, v64):
    """A workspace sized for one method is large enough for the other, and an
    FP32 one has room for method 0's checkpoints (every 8 steps)."""
    lib = G._bind()
    pr = G.HestonGreeksProblem()
    pr.dtype, pr.variance_f64, pr.paths, pr.nsteps = dtype, v64, 1000, 365
    sizes = []
    for method in (0, 1):
        pr.method = method
        sizes.append(lib.sdegpu_heston_greeks_workspace(pr))
    assert sizes[0] == sizes[1]
    if dtype == _lib.F32 and not v64:
        assert sizes[0] > 46 * 1000 * 4


@pytest.mark.parametrize('value,want', [
    (None, np.nan), (np.array(None), np.nan), ('0.25', .25), (True, 1.),
    (np.float32(.25), .25), (np.array(.25), .25), (np.ma.masked, 0.),
    (np.datetime64(3, 'D'), 3.)])
def test_scalar_parameters_convert_as_arrays_do(value, want):
    """Whatever NumPy converts to one double is a scalar parameter (None is NaN),
    as it is inside an array."""
    t0s = np.array([0., .5])
    p = sa.lognorm_process(paths=4, mu=value, steps=4)
    assert p._path_params(t0s) is None
    got = p._eval('mu', t0s, (1,))
    assert got.dtype == np.float64 and got.shape == (2, 1)
    assert np.array_equal(got, np.full((2, 1), want), equal_nan=True)
    with pytest.raises(TypeError):
        sa.lognorm_process(paths=4, mu=1j, steps=4)._eval('mu', t0s, (1,))


@pytest.mark.parametrize('model,nvars,field,want', [
    (_lib.MODEL_OU, 4, None, 65536), (_lib.MODEL_OU, 5, None, 32768),
    (_lib.MODEL_HESTON, 4, None, 65536), (_lib.MODEL_HESTON, 6, None, 16384),
    (_lib.MODEL_CIR, 1, 'replay_dw', 16384), (_lib.MODEL_LOGNORM, 4, 'nvars_total', 16384),
    (_lib.MODEL_JUMPDIFF, 2, None, 65536), (_lib.MODEL_JUMPDIFF, 8, None, 65536),
    (_lib.MODEL_JUMPDIFF, 1, 'lam_paths', 65536), (_lib.MODEL_JUMPDIFF, 1, 'replay_dj', 16384)])
def test_row_moments_are_separate_where_that_is_faster(model, nvars, field, want, monkeypatch):
    """prepare(moments=True) gives up the fused moments of small runs only where
    several waves share paths, or where the two kernels take less."""
    prob = _lib.EulerProblem()
    prob.model, prob.nvars = model, nvars
    if field:
        setattr(prob, field, 16)
    assert integ._separate_paths(prob) == want
    monkeypatch.setattr(integ, '_SEPARATE_PATHS', 0)
    assert integ._separate_paths(prob) == 0
