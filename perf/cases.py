"""Workloads of this framework, as a user's program runs them.

Five kinds of work, each through its public entry points:

* ``paths``    a preset process on a timeline: called (``x = p(tt)``, the
               result a host array) or prepared once and launched again with
               fresh draws (``run.launch(fresh=True)``, the result on the GPU);
* ``summary``  the cross-path and along-time summaries of a prepared run;
* ``heston``   price and 7 pathwise Greeks of a European option, Heston;
* ``merton``   price and 5 pathwise Greeks, lognormal / Merton;
* ``batch``    many uneven simulations in one persistent launch.

``exact`` restates the draws (Philox4x32-10 counters, Box-Muller, Poisson
inversion) and the Euler schemes in 64 bits with plain torch and numpy.
"""
import math

import numpy as np
import torch

import sdepy_amd as sa
from sdepy_amd import batched, greeks

MODELS = ('lognorm', 'ou', 'hw', 'cir', 'heston', 'merton', 'kou')


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------

def _paths(name, model, dtype, paths, steps, rows, nvar=0, corr=False,
           anti=False, how='launch'):
    c = dict(kind='paths', model=model, dtype=dtype, paths=paths, steps=steps,
             rows=rows, nvar=nvar, corr=corr, anti=anti, how=how)
    return dict(c, name=name) if name else c


def listed():
    return [
        # interactive use: a small preset called from a script or notebook in
        # sdepy's default double precision; latency and launches count
        _paths('gbm_call_small_f64', 'lognorm', 'float64', 1000, 100, 101, how='call'),
        # the 10k x 252 GBM in double precision, prepared once, simulated
        # again with fresh draws, with its row moments (repeated small runs)
        _paths('gbm_10k_moments_f64', 'lognorm', 'float64', 10_000, 252, 253, how='moments'),
        # a correlated 4-factor full path, the largest output (16 GB)
        _paths('ou4_corr_fullpath_f32', 'ou', 'float32', 1_000_000, 1000, 1001, nvar=4,
               corr=True),
        # Heston terminal values for a European payoff, as many paths as a
        # production price takes
        _paths('heston_terminal_f32', 'heston', 'float32', 4_000_000, 365, 2, corr=True),
        # Heston in the default precision at month ends, called, with its
        # diagnostics on the host
        _paths('heston_monthly_f64', 'heston', 'float64', 99_999, 360, 13, corr=True,
               how='call'),
        # jump diffusion at a few dates
        _paths('merton_quarterly_f32', 'merton', 'float32', 2_000_000, 252, 5),
        # double exponential jumps, every step stored, default precision,
        # antithetic Wiener increments
        _paths('kou_fullpath_f64', 'kou', 'float64', 60_000, 250, 251, anti=True),
        # a basket of 20 correlated assets at month ends, default precision
        _paths('basket20_monthly_f64', 'lognorm', 'float64', 100_000, 252, 13, nvar=20,
               corr=True),
        # risk run: price and 7 Greeks by the adjoint, 4M x 365
        dict(name='heston_greeks_f32', kind='heston', dtype='float32', paths=4_000_000,
             steps=365, method='adjoint', payoff='call', xi=.5),
        # price and 5 Greeks under Merton, 2M x 252
        dict(name='merton_greeks_f32', kind='merton', dtype='float32', paths=2_000_000,
             steps=252, lam=1., payoff='call'),
        # a book of 256 uneven simulations, moments of the terminal values
        dict(name='batch256_f32', kind='batch', n=256, min_paths=1000, max_paths=100_000,
             max_steps=1000, shape=7),
        # what is read off a full path: moments, extremes, a histogram
        dict(name='summary_fullpath_f32', kind='summary', dtype='float32', paths=500_000,
             steps=252),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(('paths', 'summary', 'heston', 'merton', 'batch'),
                       (8, 1, 2, 1.5, 1))[0]
    dtype = rng.choice(('float32', 'float64'))
    if kind == 'paths':
        model = rng.choice(MODELS)
        wide = model in ('lognorm', 'ou') and rng.random() < .2
        nvar = rng.randint(9, 40) if wide else rng.choice((0, 0, 0, 2, 3, 4, 5))
        if model in ('heston', 'hw') and nvar:
            nvar = rng.randint(2, 4)
        if model in ('merton', 'kou'):
            nvar = rng.choice((0, 0, 2))
        corr = model in ('hw', 'heston') or wide or (nvar > 1 and rng.random() < .7)
        how = rng.choice(('call', 'launch', 'launch', 'moments'))
        if wide and how == 'moments':
            how = 'launch'
        steps = _log_int(rng, 12, 1000)
        width = max(1, nvar) * (2 if model in ('heston', 'hw') else 1)
        top = 10_000_000 if how == 'call' else \
            600_000_000 if dtype == 'float32' else 300_000_000
        top = top // (steps * width)
        paths = _log_int(rng, 500, max(1000, min(4_000_000, top)))
        rows = rng.choice((2, 5, 13, steps + 1))
        rows = min(rows, steps + 1)
        anti = rng.random() < .25
        if anti:
            paths += paths % 2
        return _paths(None, model, dtype, paths, steps, rows, nvar, corr, anti, how)
    if kind == 'summary':
        steps = _log_int(rng, 12, 500)
        return dict(kind=kind, dtype=dtype, steps=steps,
                    paths=_log_int(rng, 1000, min(1_000_000, 150_000_000 // steps)))
    if kind == 'heston':
        steps = _log_int(rng, 12, 730)
        top = 1_400_000_000 if dtype == 'float32' else 300_000_000
        return dict(kind=kind, dtype=dtype, steps=steps,
                    paths=_log_int(rng, 10_000, min(4_000_000, top // steps)),
                    method=rng.choice(('adjoint', 'adjoint', 'tangent')),
                    payoff=rng.choice(('call', 'put')), xi=rng.choice((.2, .25, .5)))
    if kind == 'merton':
        steps = _log_int(rng, 12, 730)
        return dict(kind=kind, dtype=dtype, steps=steps,
                    paths=_log_int(rng, 10_000, min(4_000_000, 600_000_000 // steps)),
                    lam=rng.choice((0., .5, 1., 5.)), payoff=rng.choice(('call', 'put')))
    return dict(kind=kind, n=rng.randint(16, 256), min_paths=1000,
                max_paths=_log_int(rng, 5000, 100_000), max_steps=rng.randint(50, 1000),
                shape=rng.randint(0, 10 ** 6))


# --------------------------------------------------------------------------
# parameters and keys, from the seed alone
# --------------------------------------------------------------------------

def _correlation(g, m):
    a = g.standard_normal((m, m))
    s = a @ a.T + m * np.eye(m)
    d = 1 / np.sqrt(np.diag(s))
    return s * d[:, None] * d[None, :]


def _setup(case, seed):
    """Parameters, component shape and timeline of a `paths` case."""
    g = np.random.default_rng(seed)
    model, n = case['model'], case['nvar']
    vshape = (n,) if n else ()
    col = vshape + (1,)

    def u(lo, hi):
        v = g.uniform(lo, hi, col)
        return v if n else float(v[0])
    p, corr, rho = {}, None, None
    if model in ('lognorm', 'merton', 'kou'):
        p.update(x0=u(.8, 1.2), mu=u(0., .1), sigma=u(.1, .4))
    elif model == 'ou':
        p.update(x0=u(-.5, .5), theta=u(-1., 1.), k=u(.5, 3.), sigma=u(.1, .5))
    elif model == 'cir':
        p.update(x0=u(.03, .06), theta=u(.03, .06), k=u(1., 3.), xi=u(.1, .3))
    elif model == 'hw':
        f = vshape + (2, 1)
        p.update(x0=0., theta=0., k=g.uniform(.05, .5, f), sigma=g.uniform(.005, .02, f))
    else:
        p.update(x0=u(80., 120.), mu=u(0., .05), sigma=1., y0=u(.03, .06),
                 theta=u(.03, .06), k=u(1.5, 2.5), xi=u(.3, .5))
    if model == 'merton':
        p.update(lam=float(g.uniform(.5, 2.)), a=float(g.uniform(-.15, .05)),
                 b=float(g.uniform(.05, .2)))
    elif model == 'kou':
        p.update(lam=float(g.uniform(.5, 2.)), a=float(g.uniform(.05, .15)),
                 b=float(g.uniform(.05, .15)), pa=float(g.uniform(.3, .7)))
    if case['corr']:
        if model == 'heston':
            rho = float(g.uniform(-.8, -.3)) if not n else g.uniform(-.8, -.3, n)
        elif model == 'hw':
            corr = _correlation(g, 2)
        elif n:
            corr = _correlation(g, n)
    grid = np.linspace(0., 1., case['steps'] + 1)
    at = np.unique(np.round(np.linspace(0, case['steps'], case['rows'])).astype(int))
    return p, corr, rho, vshape, grid, at


CLASSES = {'lognorm': 'lognorm_process', 'ou': 'ornstein_uhlenbeck_process',
           'hw': 'hull_white_process', 'cir': 'cox_ingersoll_ross_process',
           'heston': 'full_heston_process', 'merton': 'merton_jumpdiff_process',
           'kou': 'kou_jumpdiff_process'}


def _process(case, seed):
    p, corr, rho, vshape, grid, at = _setup(case, seed)
    if case['model'] == 'hw':
        p['factors'] = 2
    info = {}
    proc = getattr(sa, CLASSES[case['model']])(
        paths=case['paths'], vshape=vshape, dtype=np.dtype(case['dtype']),
        rng=np.random.default_rng(seed + 1), steps=grid, info=info, corr=corr, rho=rho,
        dw=sa.odd_wiener_source if case['anti'] else None, **p)
    return proc, info, grid[at]


HPRM = dict(x0=100., r=.02, k=2., theta=.04, rho=-.7, y0=.04)
MPRM = dict(x0=1., mu=.03, sigma=.2, a=-.1, b=.15)


def _key(seed, which=0):
    g = np.random.default_rng(seed + 17 + which)
    return tuple(int(v) for v in g.integers(0, 2 ** 32, size=2, dtype=np.uint64))


def _summary_case(case):
    return _paths(None, 'lognorm', case['dtype'], case['paths'], case['steps'],
                  case['steps'] + 1)


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------

def prepare(case, seed):
    kind = case['kind']
    s = {'case': case}
    if kind == 'paths':
        proc, info, tt = _process(case, seed)
        s.update(proc=proc, info=info, tt=tt)
        if case['how'] != 'call':
            s['run'] = proc.prepare(tt, moments=case['how'] == 'moments')
    elif kind == 'summary':
        proc, _, tt = _process(_summary_case(case), seed)
        s['run'] = proc.prepare(tt)
        s['run'].launch()
    elif kind == 'heston':
        s['run'] = greeks.HestonGreeks(
            paths=case['paths'], steps=case['steps'], dtype=np.dtype(case['dtype']),
            strike=100., maturity=1., method=case['method'], payoff=case['payoff'],
            xi=case['xi'], key=_key(seed), **HPRM)
    elif kind == 'merton':
        s['run'] = greeks.LogGreeks(
            paths=case['paths'], steps=case['steps'], dtype=np.dtype(case['dtype']),
            strike=1., r=.03, maturity=1., lam=case['lam'], payoff=case['payoff'],
            key_w=_key(seed), key_j=_key(seed, 1), **MPRM)
    else:
        s['run'] = batched.BatchedTerminalMoments(_specs(case, seed))
    return s


def _specs(case, seed):
    shape, g = np.random.default_rng(case['shape']), np.random.default_rng(seed)
    specs = []
    for i in range(case['n']):
        paths = int(round(10 ** shape.uniform(math.log10(case['min_paths']),
                                              math.log10(case['max_paths']))))
        kw = dict(paths=paths, steps=int(shape.integers(12, case['max_steps'] + 1)),
                  dtype=np.float32, rng=np.random.default_rng(seed + 1 + i))
        if i % 2 == 0:
            p = sa.lognorm_process(x0=1., mu=g.uniform(0, .1), sigma=g.uniform(.1, .5), **kw)
        else:
            p = sa.hull_white_process(factors=2, x0=0., theta=0.,
                                      k=g.uniform(.01, .3, (2, 1)),
                                      sigma=g.uniform(.005, .02, (2, 1)),
                                      rho=g.uniform(-.9, .9), **kw)
        specs.append((p, (0., 1.)))
    return specs


def run(s):
    case = s['case']
    kind = case['kind']
    if kind == 'paths':
        if case['how'] == 'call':
            x = s['proc'](s['tt'])
            out = {'x': list(x) if isinstance(x, tuple) else [x]}
            for k in ('negative_y_count', 'jump_count', 'jump_rate'):
                if k in s['info']:
                    out[k] = s['info'][k]
            return out
        r = s['run']
        r.launch(fresh=True)
        if case['how'] == 'launch':
            return {'x': r.xx_dev}
        m, v = r.pmean(), r.pvar()
        return {'x': r.xx_dev, 'mean': list(m) if isinstance(m, tuple) else [m],
                'var': list(v) if isinstance(v, tuple) else [v]}
    if kind == 'summary':
        r = s['run']
        mc = r.montecarlo(row=-1, bins=100)
        counts, edges = mc.histogram()
        return {'mean': r.pmean(), 'var': r.pvar(), 'min': r.pmin(), 'max': r.pmax(),
                'tmax': r.tmax(), 'mc': [mc.mean(), mc.std(), mc.skew(), mc.kurtosis()],
                'counts': counts, 'edges': edges}
    if kind in ('heston', 'merton'):
        s['run'].launch()
        res = s['run'].result()
        return {'price': res.price, 'price_se': res.price_se, 'greeks': res.greeks,
                'greeks_se': res.greeks_se}
    mean, var = s['run'].run()
    return {'mean': mean, 'var': var}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

# operations per normal (its share of a Philox block and of a Box-Muller
# pair) and per step of one component
NORMAL = 22
STEP = {'lognorm': 4, 'ou': 4, 'hw': 4, 'cir': 9, 'heston': 9, 'merton': 18, 'kou': 18}


def work(case):
    kind = case['kind']
    if kind == 'paths':
        es = np.dtype(case['dtype']).itemsize
        n = max(1, case['nvar'])
        m = n * (2 if case['model'] in ('heston', 'hw') else 1)
        out = n * (2 if case['model'] == 'heston' else 1)
        rows = min(case['rows'], case['steps'] + 1)
        per = m * (NORMAL / (2 if case['anti'] else 1) + STEP[case['model']])
        if case['corr']:
            per += n * 4 if case['model'] in ('heston', 'hw') else m * (m + 1)
        return {'bytes': rows * out * case['paths'] * es,
                'flops': case['paths'] * case['steps'] * per}
    if kind == 'summary':
        es = np.dtype(case['dtype']).itemsize
        n = case['paths'] * (case['steps'] + 1)
        return {'bytes': n * es + case['paths'] * es, 'flops': 6 * n}
    if kind == 'heston':
        # generator, Euler step, partial derivatives of one variance
        return {'bytes': 16 * 8, 'flops': case['paths'] * case['steps'] * (2 * NORMAL + 46)}
    if kind == 'merton':
        jump = 12 if case['lam'] else 0
        return {'bytes': 12 * 8, 'flops': case['paths'] * case['steps'] * (NORMAL + 2 + jump)}
    shape = np.random.default_rng(case['shape'])
    total = 0
    for i in range(case['n']):
        paths = int(round(10 ** shape.uniform(math.log10(case['min_paths']),
                                              math.log10(case['max_paths']))))
        steps = int(shape.integers(12, case['max_steps'] + 1))
        total += paths * (steps - 1) * (NORMAL + 3 if i % 2 == 0 else 2 * NORMAL + 10)
    return {'bytes': case['n'] * 16, 'flops': total}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------

MASK = 0xFFFFFFFF


def _philox(c0, path, c2, c3, key):
    """Philox4x32-10 (Salmon et al. 2011) of counter (c0, path, c2, c3), c0 a
    number or a tensor: four int64 tensors of 32-bit words."""
    x = [torch.as_tensor(c0, dtype=torch.int64, device=path.device) + 0 * path, path,
         torch.full_like(path, c2), torch.full_like(path, c3)]
    k0, k1 = key
    for _ in range(10):
        # the 64-bit products wrap as unsigned ones do; >> is masked below
        p0, p1 = x[0] * 0xD2511F53, x[2] * 0xCD9E8D57
        x = [((p1 >> 32) & MASK) ^ x[1] ^ k0, p1 & MASK,
             ((p0 >> 32) & MASK) ^ x[3] ^ k1, p0 & MASK]
        k0, k1 = (k0 + 0x9E3779B9) & MASK, (k1 + 0xBB67AE85) & MASK
    return x


def _u01(w):
    return (w.double() + .5) * 2. ** -32


def _block_normals(w):
    z = []
    for a, b in ((w[0], w[1]), (w[2], w[3])):
        r, ang = torch.sqrt(-2 * torch.log(_u01(a))), 2 * math.pi * _u01(b)
        z += [r * torch.cos(ang), r * torch.sin(ang)]
    return z


class _Stream:
    """Values g = 0, 1, ... of a path's stream, four to a block."""

    def __init__(self, path, c2, epoch, key, normal):
        self.path, self.c2, self.epoch, self.key = path, c2, epoch, key
        self.normal, self.have = normal, {}

    def __call__(self, g):
        b = g // 4
        if b not in self.have:
            w = _philox(b, self.path, self.c2, self.epoch, self.key)
            self.have = {b: _block_normals(w) if self.normal else w}
        return self.have[b][g % 4]


def _poisson(word, lam):
    """Counts by sequential inversion of the distribution function."""
    u = _u01(word)
    n = torch.zeros_like(word)
    p = f = torch.full_like(u, math.exp(-lam))
    k = 0
    more = u > f
    while bool(more.any()) and k < 4096:
        k += 1
        p = p * (lam / k)
        n = torch.where(more, n + 1, n)
        f = torch.where(more, f + p, f)
        more = more & (u > f)
    return n


def _jump_sizes(model, prm, n, path, slot, epoch, key):
    """Sums of n jump sizes of each path at a slot."""
    total = torch.zeros(path.shape, dtype=torch.float64, device=path.device)
    at = torch.nonzero(n).reshape(-1)
    if at.numel():
        cnt, who = n[at], path[at]
        acc = torch.zeros(at.shape, dtype=torch.float64, device=path.device)
        per = 4 if model == 'merton' else 2
        for j in range(int(cnt.max())):
            if j % per == 0:
                w = _philox(slot, who, 2 | (j // per) << 8, epoch, key)
                z = _block_normals(w) if model == 'merton' else None
            if model == 'merton':
                y = prm['a'] + prm['b'] * z[j % 4]
            else:
                up = _u01(w[2 * (j % 2) + 1]) <= prm['pa']
                e = -torch.log(_u01(w[2 * (j % 2)]))
                y = torch.where(up, prm['a'] * e, -prm['b'] * e)
            acc = torch.where(cnt > j, acc + y, acc)
        total[at] = acc
    return total


def _simulate(case, seed, epoch):
    """Stored rows [rows][values][paths] in 64 bits, and the counts kept."""
    prm, corr, rho, vshape, grid, at = _setup(case, seed)
    model, n, P = case['model'], max(1, case['nvar']), case['paths']
    g = np.random.default_rng(seed + 1)
    key = tuple(int(v) for v in g.integers(0, 2 ** 32, size=2, dtype=np.uint64))
    key_j = tuple(int(v) for v in g.integers(0, 2 ** 32, size=2, dtype=np.uint64))
    dev = torch.device('cuda')
    path = torch.arange(P, dtype=torch.int64, device=dev)
    sign = 1.
    path_w = path
    if case['anti']:
        path_w = torch.where(path < P // 2, path, path - P // 2)
        sign = torch.where(path < P // 2, 1., -1.).double()
    wide = model in ('heston', 'hw')
    M = n * (2 if wide else 1)
    if model == 'heston' and rho is not None:
        r = np.broadcast_to(rho, n)
        corr = np.block([[np.eye(n), np.diag(r)], [np.diag(r), np.eye(n)]])
    L = np.eye(M)
    if corr is not None:
        L = np.kron(np.eye(M // corr.shape[0]), np.linalg.cholesky(corr))

    def vec(name, m=n):
        return np.broadcast_to(np.asarray(prm[name], float).reshape(-1), m)
    if model == 'hw':
        x = [torch.zeros(P, dtype=torch.float64, device=dev) for _ in range(M)]
    else:
        x = [torch.full((P,), float(v), dtype=torch.float64, device=dev) for v in vec('x0')]
        if model in ('lognorm', 'merton', 'kou', 'heston'):
            x = [torch.log(v) for v in x]
        if model == 'heston':
            x += [torch.full((P,), float(v), dtype=torch.float64, device=dev)
                  for v in vec('y0')]
    log = model in ('lognorm', 'merton', 'kou')
    nout = n * (2 if model == 'heston' else 1)
    out = torch.empty((at.size, nout, P), dtype=torch.float64, device=dev)
    counts = [torch.zeros(P, dtype=torch.int64, device=dev) for _ in range(n)]

    def store(row):
        if model == 'hw':
            vals = [x[2 * i] + x[2 * i + 1] for i in range(n)]
        elif model == 'heston':
            vals = [torch.exp(v) for v in x[:n]] + x[n:]
        else:
            vals = [torch.exp(v) for v in x] if log else x
        for i, v in enumerate(vals):
            out[row, i] = v
    rows = {int(s): i for i, s in enumerate(at)}
    if 0 in rows:
        store(rows[0])
    zs = _Stream(path_w, 0, epoch, key, True)
    ns = _Stream(path, 1, epoch, key_j, False)
    for s in range(case['steps']):
        ds = float(grid[s + 1] - grid[s])
        sq = math.sqrt(ds)
        z = [zs(s * M + v) * sign for v in range(M)]
        dw = []
        for i in range(M):
            acc = None
            for j in range(i + 1):
                if L[i, j]:
                    t = z[j] * (float(L[i, j]) * sq)
                    acc = t if acc is None else acc + t
            dw.append(acc)
        for i in range(n if model != 'hw' else M):
            if model in ('lognorm', 'merton', 'kou'):
                mu, sig = float(vec('mu')[i]), float(vec('sigma')[i])
                inc = dw[i] * sig + (mu - sig * sig / 2) * ds
                if model != 'lognorm':
                    slot = s * M + i
                    cnt = _poisson(ns(slot), prm['lam'] * ds)
                    inc = inc + _jump_sizes(model, prm, cnt, path, slot, epoch, key_j)
                    counts[i] += cnt
                x[i] = x[i] + inc
            elif model in ('ou', 'hw'):
                k, th, sig = (float(vec(q, M)[i]) for q in ('k', 'theta', 'sigma'))
                x[i] = x[i] + (k * (th - x[i]) * ds + sig * dw[i])
            elif model == 'cir':
                k, th, xi = (float(vec(q)[i]) for q in ('k', 'theta', 'xi'))
                xp = torch.clamp(x[i], min=0.)
                x[i] = x[i] + (k * (th - xp) * ds + xi * torch.sqrt(xp) * dw[i])
            else:
                mu, sig, k, th, xi = (float(vec(q)[i])
                                      for q in ('mu', 'sigma', 'k', 'theta', 'xi'))
                y = x[n + i]
                counts[i] += y < 0
                yp = torch.clamp(y, min=0.)
                sy = torch.sqrt(yp)
                x[i] = x[i] + ((mu - sig * sig * yp / 2) * ds + sig * sy * dw[i])
                x[n + i] = y + (k * (th - yp) * ds + xi * sy * dw[n + i])
        if s + 1 in rows:
            store(rows[s + 1])
    return out, counts, vshape


def _exact_paths(case, seed):
    out, counts, vshape = _simulate(case, seed, 0 if case['how'] == 'call' else 1)
    if case['how'] == 'call':
        n = max(1, case['nvar'])
        parts = [out[:, :n], out[:, n:]] if case['model'] == 'heston' else [out]
        res = {'x': [q.reshape((q.shape[0],) + vshape + (q.shape[-1],)) for q in parts]}
        if case['model'] == 'heston':
            res['negative_y_count'] = None
        elif case['model'] in ('merton', 'kou'):
            res.update(jump_count=None, jump_rate=None)
        return res
    if case['how'] == 'launch':
        return {'x': out}
    n = max(1, case['nvar'])
    parts = [out[:, :n], out[:, n:]] if case['model'] == 'heston' else [out]
    shape = (out.shape[0],) + vshape + (1,)
    return {'x': out, 'mean': [q.mean(-1).reshape(shape) for q in parts],
            'var': [q.var(-1, correction=0).reshape(shape) for q in parts]}


def _option(S, payoff, strike, disc):
    intr = S - strike if payoff == 'call' else strike - S
    itm = intr > 0
    pay = torch.where(itm, disc * intr, 0.)
    xbar = torch.where(itm, disc * S if payoff == 'call' else -disc * S, 0.)
    return pay, xbar


def _with_errors(pay, g):
    def se(v):
        return float(torch.sqrt(v.var(correction=0) / (v.numel() - 1)))
    return {'price': float(pay.mean()), 'price_se': se(pay),
            'greeks': {k: float(v.mean()) for k, v in g.items()},
            'greeks_se': {k: se(v) for k, v in g.items()}}


def _exact_heston(case, seed):
    """Derivatives carried along the full-truncation Euler scheme.  With
    xi = .5 (2 k theta < xi^2) the variance reaches 0 and single paths
    dominate the sums of 1 / sqrt(v), so that no rounding determines the
    variance's Greeks to a digit: there they have no value here."""
    p, n, P = dict(HPRM, xi=case['xi']), case['steps'], case['paths']
    path = torch.arange(P, dtype=torch.int64, device='cuda')
    zs = _Stream(path, 0, 0, _key(seed), True)
    grid = np.linspace(0., 1., n + 1)
    rho, rc = p['rho'], math.sqrt(1 - p['rho'] ** 2)
    X = torch.full((P,), math.log(p['x0']), dtype=torch.float64, device='cuda')
    V = torch.full_like(X, p['y0'])
    dV = {q: torch.zeros_like(X) for q in ('k', 'theta', 'xi', 'rho')}
    dV['y0'] = torch.ones_like(X)
    dX = {q: torch.zeros_like(X) for q in dV}
    for s in range(n):
        ds = float(grid[s + 1] - grid[s])
        sq = math.sqrt(ds)
        z0, z1 = zs(2 * s), zs(2 * s + 1)
        w = rho * z0 + rc * z1
        pos = V > 0
        vp = torch.clamp(V, min=0.)
        sv = torch.sqrt(vp)
        half = torch.where(pos, .5 / torch.where(pos, sv, 1.), 0.)
        a = torch.where(pos, 1 - p['k'] * ds + p['xi'] * sq * w * half, 1.)
        b = torch.where(pos, -.5 * ds + sq * z0 * half, 0.)
        src = {'k': (p['theta'] - vp) * ds, 'theta': p['k'] * ds, 'xi': sv * sq * w,
               'rho': p['xi'] * sv * sq * (z0 - rho / rc * z1), 'y0': 0.}
        for q in dV:
            dX[q] = dX[q] + b * dV[q]
            dV[q] = a * dV[q] + src[q]
        X = X + ((p['r'] - .5 * vp) * ds + sv * sq * z0)
        V = V + (p['k'] * (p['theta'] - vp) * ds + p['xi'] * sv * sq * w)
    S = torch.exp(X)
    pay, xbar = _option(S, case['payoff'], 100., math.exp(-p['r']))
    g = {'x0': xbar / p['x0'], 'r': xbar - pay}
    g.update({q: xbar * dX[q] for q in dX})
    res = _with_errors(pay, g)
    if case['xi'] > .3:
        for part in ('greeks', 'greeks_se'):
            res[part].update({q: None for q in dX})
    return res


def _exact_merton(case, seed):
    p, n, P, lam = MPRM, case['steps'], case['paths'], case['lam']
    path = torch.arange(P, dtype=torch.int64, device='cuda')
    zs = _Stream(path, 0, 0, _key(seed), True)
    ns = _Stream(path, 1, 0, _key(seed, 1), False)
    grid = np.linspace(0., 1., n + 1)
    sdw = torch.zeros(P, dtype=torch.float64, device='cuda')
    sz = torch.zeros_like(sdw)
    nj = torch.zeros_like(path)
    for s in range(n):
        ds = float(grid[s + 1] - grid[s])
        sdw = sdw + math.sqrt(ds) * zs(s)
        if lam:
            cnt = _poisson(ns(s), lam * ds)
            nj += cnt
            sz = sz + _jump_sizes('merton', {'a': 0., 'b': 1.}, cnt, path, s, 0, _key(seed, 1))
    x = math.log(p['x0']) + (p['mu'] - p['sigma'] ** 2 / 2) + p['sigma'] * sdw + \
        p['a'] * nj + p['b'] * sz
    S = torch.exp(x)
    pay, xbar = _option(S, case['payoff'], 1., math.exp(-.03))
    return _with_errors(pay, {'x0': xbar / p['x0'], 'mu': xbar,
                              'sigma': xbar * (sdw - p['sigma']), 'a': xbar * nj,
                              'b': xbar * sz})


def _exact_summary(case, seed):
    x = _simulate(_summary_case(case), seed, 0)[0][:, 0]
    shape = (x.shape[0], 1)
    last = x[-1]
    m, v = last.mean(), last.var(correction=0)
    d = last - m
    skew, kurt = (d ** 3).mean() / v ** 1.5, (d ** 4).mean() / v ** 2
    return {'mean': x.mean(-1).reshape(shape), 'var': x.var(-1, correction=0).reshape(shape),
            'min': x.amin(-1).reshape(shape), 'max': x.amax(-1).reshape(shape),
            'tmax': x.amax(0).reshape(1, -1),
            'mc': [float(m), float(torch.sqrt(v)), float(skew), float(kurt)],
            'counts': None, 'edges': None}


def exact(case, seed):
    kind = case['kind']
    if kind == 'paths':
        return _exact_paths(case, seed)
    if kind == 'heston':
        return _exact_heston(case, seed)
    if kind == 'merton':
        return _exact_merton(case, seed)
    if kind == 'summary':
        return _exact_summary(case, seed)
    # a batch is some hundred thousand steps: too long here
    return None
