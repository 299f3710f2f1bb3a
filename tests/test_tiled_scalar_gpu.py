"""The tiled scalar march (k_st_tiled of spacetime.hip) against the oracle,
value for value: rings shorter than a wavefront's overlap, than a window and
longer, launches and exchanges that end anywhere, and values that leave the
range of its shared reciprocals.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(orc, kind, ncelm, dt=0.4, nvar=1):
    from solvcon_amd import spacetime as st
    rng = np.random.default_rng(ncelm)
    g = st.Grid(np.cumsum(rng.uniform(0.5, 1.5, ncelm + 1)))
    ids = {'default': orc.ST_DEFAULT, 'linear': orc.ST_LINEAR,
           'burgers': orc.ST_BURGERS}
    if kind == 'default':
        s = st.Solver(grid=g, time_increment=dt, nvar=nvar)
    elif kind == 'linear':
        s = st.LinearScalarSolver(grid=g, time_increment=dt)
    else:
        s = st.InviscidBurgersSolver(grid=g, time_increment=dt)
    o = orc.StSolver(ids[kind], g.xcoord.ndarray, dt, nvar)
    u, ux = rng.uniform(-1, 1, (2, g.xsize, nvar))
    for e in (s, o):
        (e.so0.ndarray if e is s else e.so0)[...] = u
        (e.so1.ndarray if e is s else e.so1)[...] = ux
        e.setup_march()
    return s, o


def _same(s, o):
    for t in ('so0', 'so1', 'cfl'):
        assert np.array_equal(getattr(s, t).ndarray, getattr(o, t),
                              equal_nan=True), t


# A window is 196 elements, a wavefront's overlap 10; rings of up to 32
# elements run 24 steps per launch, of 20001 and more too, others 64.  One block
# alone on its ring marches in place: up to 186 elements for one step, 184 for
# two, 56 for 64.
@pytest.mark.parametrize('ncelm,steps', [
    (1, 50), (2, 2), (8, 49), (9, 48), (10, 17), (30, 47), (31, 130), (54, 128),
    (64, 129), (100, 3), (188, 127), (195, 64), (300, 257), (19998, 70),
    (54, 64), (55, 64), (184, 1), (185, 1), (182, 2), (183, 2), (31, 24),
    (19999, 49), (40000, 25)])
@pytest.mark.parametrize('kind,alpha', [('linear', 2), ('burgers', 1),
                                        ('burgers', 2)])
def test_tiled_scalar_sizes(orc, ncelm, steps, kind, alpha):
    print('case: tiled scalar', ncelm, steps, kind, alpha, flush=True)
    s, o = _pair(orc, kind, ncelm)
    for k in (steps, 1):
        getattr(s, 'march_alpha%d' % alpha)(k)
        o.march(alpha, k)
        _same(s, o)


@pytest.mark.parametrize('val', [0.0, 1e-120, -3e-310, 1e80, np.inf, np.nan])
@pytest.mark.parametrize('kind', ['linear', 'burgers'])
@pytest.mark.parametrize('ncelm', [20, 500])
def test_tiled_scalar_out_of_range(orc, ncelm, kind, val):
    # Everywhere but one stretch (quotients of tiny values all over), and in
    # single elements beside the seam and inside.
    print('case: tiled scalar out of range', ncelm, kind, val, flush=True)
    s, o = _pair(orc, kind, ncelm)
    with np.errstate(all='ignore'):
        for a, b in ((s.so0.ndarray, s.so1.ndarray), (o.so0, o.so1)):
            if abs(val) < 1e-100:
                a[10:] *= val
                b[10:] *= val
            else:
                a[[2, 12, 2 * ncelm + 2]] = val
                b[8] = val
        s.march_alpha2(20)
        o.march(2, 20)
        _same(s, o)


# A time increment far beyond the stable one: values grow from within the range
# out of it, between two exchanges and at different steps in each wavefront.
@pytest.mark.parametrize('kind', ['linear', 'burgers'])
@pytest.mark.parametrize('ncelm,dt', [(7, 9.0), (20, 9.0), (500, 3.0), (500, 30.0)])
def test_tiled_scalar_leaves_range(orc, ncelm, dt, kind):
    print('case: tiled scalar leaves range', ncelm, dt, kind, flush=True)
    s, o = _pair(orc, kind, ncelm, dt=dt)
    with np.errstate(all='ignore'):
        for k in (6, 13, 22):
            s.march_alpha2(k)
            o.march(2, k)
            _same(s, o)


@pytest.mark.parametrize('ncelm', [77, 400])
@pytest.mark.parametrize('nvar', [1, 3])
def test_tiled_scalar_variables(orc, ncelm, nvar):
    # Only variable 0 is marched; the others and the outermost rows stay,
    # through calls of odd and even numbers of launches.
    print('case: tiled scalar', ncelm, nvar, 'variables', flush=True)
    s, o = _pair(orc, 'default', ncelm, nvar=nvar)
    for steps in (66, 1, 2, 130, 64):
        s.march_alpha2(steps)
        o.march(2, steps)
        _same(s, o)


def test_tiled_scalar_clone_after_odd_launches(orc):
    # The arrays of the state have changed places: a clone and the stage calls
    # take the right ones.
    print('case: tiled scalar, clone', flush=True)
    s, o = _pair(orc, 'burgers', 400)
    s.march_alpha2(3)
    o.march(2, 3)
    c = s.clone()
    _same(c, o)
    c.march_alpha2(5)
    _same(s, o)
    s.march_half_so0(odd_plane=False)
    s.treat_boundary_so0()
    o.march_half_so0(False)
    o.treat_boundary_so0()
    assert np.array_equal(s.so0.ndarray, o.so0)
    s.march_alpha2(4)
    o.march(2, 4)
    _same(s, o)


@pytest.mark.parametrize('kind', ['default', 'linear', 'burgers'])
@pytest.mark.parametrize('ncelm', [20, 500])
def test_tiled_scalar_zero_signs(orc, ncelm, kind):
    # Zeros of both signs in most places: their signs are the oracle's too.
    print('case: tiled scalar zero signs', ncelm, kind, flush=True)
    for dt in (0.0, 0.5):
        s, o = _pair(orc, kind, ncelm, dt=dt)
        rng = np.random.default_rng(ncelm)
        n = s.so0.ndarray.shape[0]
        u, ux = rng.choice([0.0, -0.0, 0.0, -0.0, 1.0, -1.0], (2, n, 1))
        for e in (s, o):
            (e.so0.ndarray if e is s else e.so0)[...] = u
            (e.so1.ndarray if e is s else e.so1)[...] = ux
            e.setup_march()
        for steps in (2, 3):
            s.march_alpha2(steps)
            o.march(2, steps)
            for t in ('so0', 'so1', 'cfl'):
                a = np.array(getattr(s, t).ndarray)
                b = np.array(getattr(o, t))
                assert np.array_equal(a.view(np.int64), b.view(np.int64)), t
