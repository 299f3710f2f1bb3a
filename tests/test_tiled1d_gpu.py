"""The tiled 1D march (k_march_tiled of onedim.hip) against the oracle, value
for value, at the sizes where its windows, wavefronts and launches end and on
states that leave the range of its shared reciprocals.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(orc, n, dt, gamma=1.4, stretch=0.0):
    from solvcon_amd.onedim import Euler1DCore
    c, o = Euler1DCore(ncoord=n, time_increment=dt), orc.Euler1D(n, dt)
    rng = np.random.default_rng(n)
    x = np.linspace(-1.0, 1.0, n)
    if n > 5:
        h = 2.0 / (n - 1)
        x[1:-1] += stretch * h * rng.uniform(-1, 1, n - 2)
    st = np.stack([np.where(x < 0, 1.0, 0.125), np.zeros(n),
                   np.where(x < 0, 2.5, 0.25)], 1)
    st[:, 0] += 0.01 * rng.uniform(size=n)
    for e in (c, o):
        e.coord[...] = x
        e.gamma[...] = gamma
        e.so0[...] = st
        e.so1[...] = 0.0
        e.cfl[...] = 0.0
        e.setup_march()
    return c, o


def _same(c, o):
    for t in ('so0', 'so1', 'cfl'):
        assert np.array_equal(getattr(c, t), getattr(o, t), equal_nan=True), t


# One window of overlapping wavefronts is 416 rows (wavefronts of 64 elements
# 48 apart), one of consecutive ones 512; the second starts at 40001 points
# and 16 steps per launch at 60001.
@pytest.mark.parametrize('n,steps,alpha', [
    (5, 5, 1), (7, 9, 2), (95, 17, 2), (97, 17, 1), (127, 8, 2),
    (129, 20, 2), (223, 33, 2), (319, 64, 1), (415, 70, 2), (417, 63, 2),
    (419, 64, 2), (573, 65, 1), (727, 130, 2), (2001, 129, 2),
    (39999, 65, 2), (40001, 65, 1), (40003, 130, 2), (60001, 33, 2),
    (60003, 17, 1)])
def test_tiled_sizes(orc, n, steps, alpha):
    print('case: tiled march', n, steps, alpha, flush=True)
    c, o = _pair(orc, n, 0.4 / max(n - 1, 10), stretch=0.2)
    for k in (steps, 1):
        getattr(c, 'march_alpha%d' % alpha)(k)
        o.march(alpha, k)
        _same(c, o)


# Values beyond what the shared reciprocals cover, in single points: the
# wavefronts that hold them divide, infinities and NaNs included.
@pytest.mark.parametrize('which,val', [
    (0, 1e15), (0, 0.0), (0, 1e-60), (1, 1e-300), (1, -3e-310), (1, 1e90),
    (2, 1e-290), (2, np.inf), (1, np.nan)])
@pytest.mark.parametrize('n', [401, 1501])
def test_tiled_out_of_range(orc, n, which, val):
    print('case: tiled out of range', n, which, val, flush=True)
    c, o = _pair(orc, n, 0.1 / n)
    with np.errstate(all='ignore'):
        for e in (c, o):
            for at in (2, n // 2, n - 3):
                e.so0[at, which] = val
            e.so1[n // 3, which] = val
        c.march_alpha2(12)
        o.march(2, 12)
        _same(c, o)


# A time increment beyond the stable one: values grow from within the range out
# of it, between two exchanges and at different steps in each wavefront.
@pytest.mark.parametrize('n', [401, 1501, 40001])
@pytest.mark.parametrize('cfl', [2.0, 6.0])
def test_tiled_leaves_range(orc, n, cfl):
    print('case: tiled leaves range', n, cfl, flush=True)
    c, o = _pair(orc, n, cfl / (n - 1))
    with np.errstate(all='ignore'):
        for k in (6, 13, 22):
            c.march_alpha2(k)
            o.march(2, k)
            _same(c, o)


# Values out of range at first and in it again later: wavefronts divide for some
# exchanges and go back to the shared reciprocals.
@pytest.mark.parametrize('n', [401, 2001, 39999])
def test_tiled_returns_to_range(orc, n):
    print('case: tiled returns to range', n, flush=True)
    c, o = _pair(orc, n, 0.4 / (n - 1))
    for e in (c, o):
        e.so0[n // 4:3 * n // 4, 1] = 1e-300
    for k in (7, 30, 64):
        c.march_alpha2(k)
        o.march(2, k)
        _same(c, o)


@pytest.mark.parametrize('gamma', [1.0, 1.0 + 1e-9, 3.0, 1e8])
def test_tiled_gamma(orc, gamma):
    # Coefficients of gamma that vanish, and ones out of range.
    print('case: tiled gamma', gamma, flush=True)
    c, o = _pair(orc, 601, 1e-5, gamma=gamma)
    c.march_alpha2(20)
    o.march(2, 20)
    _same(c, o)


def _same_bits(c, o):
    for t in ('so0', 'so1', 'cfl'):
        a, b = np.array(getattr(c, t)), np.array(getattr(o, t))
        ok = ~np.isnan(b)
        assert np.array_equal(np.isnan(a), ~ok), t
        assert np.array_equal(a[ok].view(np.int64), b[ok].view(np.int64)), t


# Zeros of both signs in most places, on both directions of the coordinate and
# beside negative densities: their signs are the oracle's too.
@pytest.mark.parametrize('n', [201, 2001, 40001])
@pytest.mark.parametrize('gamma', [1.0, 1.4, 3.0])
@pytest.mark.parametrize('case', ['plain', 'descending', 'negative'])
def test_tiled_zero_signs(orc, n, gamma, case):
    from solvcon_amd.onedim import Euler1DCore
    print('case: tiled zero signs', n, gamma, case, flush=True)
    rng = np.random.default_rng(5)
    zero = [0.0, -0.0]
    x = np.cumsum(rng.choice([1.0, 1.5, 2.0], n))
    st = np.stack([rng.choice([1.0, 2.0], n), rng.choice(zero, n),
                   rng.choice(zero + [1.0], n)], 1)
    sx = rng.choice(zero, (n, 3))
    k = rng.random((n, 3)) < 0.1
    sx[k] = rng.choice([1.0, -1.0], k.sum())
    if case == 'descending':
        x = x[::-1].copy()
    if case == 'negative':
        st[rng.integers(0, n, 3), 0] = -1.0
    with np.errstate(all='ignore'):
        for steps in (1, 2, 9):
            c = Euler1DCore(ncoord=n, time_increment=0.5)
            o = orc.Euler1D(n, 0.5)
            for e in (c, o):
                e.coord[...] = x
                e.gamma[...] = gamma
                e.so0[...] = st
                e.so1[...] = sx
                e.cfl[...] = 0.0
                e.setup_march()
            c.march_alpha2(steps)
            o.march(2, steps)
            _same_bits(c, o)
