"""The FP64 Box-Muller transform (Gauss<double> in csrc/philox.hpp) and its
tables (csrc/gauss_tables.hpp), against 80-bit arithmetic."""
import os
import re

import numpy as np
import pytest

import sdepy_amd as sa
from oracle import philox as px

LD = np.longdouble
PI = LD('3.14159265358979323846264338327950288')
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    'sdepy_amd', 'csrc')


def _tables():
    text = open(os.path.join(CSRC, 'gauss_tables.hpp')).read()
    num = r'(-?0x[0-9a-f.]+p[+-]\d+)'
    log = re.findall(r'\{' + num + ', ' + num + r'\},', text)
    trig = re.findall(r'\{' + num + ', ' + num + r', (0x[0-9a-f]+)u, ', text)
    return (np.array([[float.fromhex(v) for v in r] for r in log]),
            np.array([[float.fromhex(r[0]), float.fromhex(r[1])] for r in trig]),
            np.array([int(r[2], 16) for r in trig], dtype=np.int64))


def _radians(words):
    """2 pi words / 2^32 reduced to (-pi/4, pi/4], and the quadrant."""
    q = (words + (1 << 29)) >> 30
    return 2 * PI * ((words - (q << 30)).astype(LD) / LD(2) ** 32), q & 3


def _cos_sin(words, half):
    a, q = _radians(words)
    a = a + PI * LD(half) / LD(2) ** 32 * 2
    c, s = np.cos(a), np.sin(a)
    return (np.choose(q, (c, -s, -c, s)), np.choose(q, (s, c, -s, -c)))


def test_tables_hold_what_they_say():
    log, trig, n = _tables()
    assert log.shape == (128, 2) and trig.shape == (64, 2)
    inv = -log[:, 0].astype(LD) / 2
    # 28-bit reciprocals near each interval's centre, so that fma(z, -2/c, 2)
    # is exact and small; entries that are multiples of 2^-44
    assert np.all(np.ldexp(inv.astype(float), 28) % 1 == 0)
    assert np.all(np.ldexp(log[:, 1], 44) % 1 == 0)
    assert np.max(np.abs(log[:, 1] - 2 * np.log(inv))) < 2. ** -56
    edges = (0x3fe60000 + (np.arange(129, dtype=np.int64) << 13) << 32).view(np.float64)
    for z in (edges[:-1], edges[1:]):
        assert np.max(np.abs(2 - 2 * z * inv.astype(float))) < 2. ** -6.97
    assert edges[80] == 1. and tuple(log[79]) == (-2., 0.)
    # sector angles whose cosines and sines are FP64 numbers to 2^-9 ulp
    assert np.max(np.abs(n - (np.arange(64) << 26))) <= 1 << 18
    for got, want in zip(trig.T, _cos_sin(n, 0)):
        assert np.max(np.abs(got - want) / np.spacing(np.maximum(np.abs(got), 1e-3))) < 2. ** -8


@pytest.mark.gpu
@pytest.mark.parametrize('paths', [1, 257, 40_000])
def test_normals_match_80_bit_arithmetic(gpu, paths):
    """Every normal of a source within 5 ulp (radius 1.8, angle 2.3, product
    0.5): all table rows, signs and the tails the draws reach."""
    slots = 5 if paths < 1000 else 64
    src = sa.wiener_source(paths=paths, vshape=(4,), rng=np.random.default_rng(5))
    z = src(np.zeros(slots), np.ones(slots))
    w = px.stream_words(src.key, 0, px.STREAM_NORMAL, slots, 4, np.arange(paths))
    w = w.astype(np.int64).reshape(slots, 2, 2, paths)
    a, b = w[:, :, 0], w[:, :, 1]
    # ln u from 1 - u where u > 1/2, both exact
    u = (a.astype(LD) + LD(.5)) / LD(2) ** 32
    near = -np.log1p(-((LD(2) ** 32 - a) - LD(.5)) / LD(2) ** 32)
    r = np.sqrt(2 * np.where(a >= 1 << 31, near, -np.log(u)))
    c, s = _cos_sin(b, .5)
    want = np.stack((r * c, r * s), axis=2).reshape(slots, 4, paths)
    assert np.max(np.abs(z - want) / np.abs(want)) <= 5 * 2. ** -52
