"""The face-lane form of the march (euler_lane.hip) against the oracle, value
for value, where its blocks and cell groups end and where it falls back to
the exact form.

Meshes with at most lane_cells cells of every type take it by themselves; 'f3'
in 2D and 'f2' in 3D name it.  A block holds 64 triangles, quadrilaterals or tetrahedra and
32 hexahedra, prisms or pyramids.
"""

import numpy as np
import pytest

import meshdefs as MD
import pair

pytestmark = pytest.mark.gpu

GAMMA = 1.4


def _defn(name):
    from solvcon_amd.gen import mixed_mesh_def, rect_mesh_def
    kind, size = name.split('-')
    if kind in ('tri', 'quad'):
        nx, ny = (int(c) for c in size.split('x'))
        return rect_mesh_def(nx, ny, kind=kind, seed=3, jitter=0.2)
    if kind == 'hex':
        n = [int(c) for c in size.split('x')]
        return MD.hex_block(*n, jitter=0.2, seed=5)
    if kind == 'both':  # triangles and quadrilaterals, uneven counts
        a = rect_mesh_def(7, 5, extent=(1.0, 1.0), kind='quad')
        cl, tp = a[3], a[2].copy()
        out, types = [], []
        for k, row in enumerate(cl):
            if k % 3 == 0:
                _, p, q, r, s = row
                out += [(3, p, q, r, 0), (3, p, r, s, 0)]
                types += [4, 4]
            else:
                out.append(tuple(row))
                types.append(tp[k])
        return 2, a[1], np.array(types, np.int32), np.array(out, np.int32)
    return mixed_mesh_def(int(size), seed=3)


def _pair(orc, defn, dt):
    import solvcon_amd as sc
    g, o = pair.gpu_mesh(defn), pair.orc_mesh(orc, defn)
    ge, oe = sc.EulerCore(mesh=g, time_increment=dt), orc.Euler(o, dt)
    rng = np.random.default_rng(8)
    n, nd = ge.ncell, ge.ndim
    st = np.zeros((n, nd + 2))
    st[:, 0] = rng.uniform(0.5, 1.5, n)
    st[:, 1:-1] = rng.uniform(-0.2, 0.2, (n, nd))
    st[:, -1] = rng.uniform(2.0, 3.0, n)
    ng = ge.ngstcell
    for e in (ge, oe):
        e.init_solution(GAMMA, 1.0, [0.0] * nd, 1.0)
    ge.so0n.ndarray[ng:] = st
    oe.so0n[ng:] = st
    f = list(o.bndfcs[:, 0])
    val = [1.05] + [0.2, 0.0, 0.0][:nd] + [1.0, GAMMA]
    for kind, faces, v in (('nonrefl', f[0::3], ()), ('slipwall', f[1::3], ()),
                           ('inlet', f[2::3], val)):
        if kind == 'inlet':
            ge.add_inlet(faces, value=v)
            oe.add_bc(orc.BC_INLET, faces, v)
        else:
            getattr(ge, 'add_' + kind)(faces)
            oe.add_bc(getattr(orc, 'BC_' + kind.upper()), faces)
    ge.bc_soln()
    ge.bc_dsoln()
    oe.call('bc_soln')
    oe.call('bc_dsoln')
    return ge, oe


NAMES = ['tri-1x1', 'tri-31x1', 'tri-8x4', 'tri-11x3', 'tri-13x5',
         'quad-63x1', 'quad-8x8', 'quad-13x5', 'hex-31x1x1', 'hex-4x4x2',
         'hex-11x3x1', 'both-0', 'mixed-4', 'mixed-7']


@pytest.mark.parametrize('name', NAMES)
def test_lane_march(orc, monkeypatch, name):
    # Chosen by itself; a normal march runs no exact pass.  Then a cell beyond
    # the fast form's range and one infinity: the wavefronts that meet them
    # take the exact form, NaNs in the oracle's places.
    print('case: lane march', name, flush=True)
    monkeypatch.delenv('SC_EULER_FORM', raising=False)
    ge, oe = _pair(orc, _defn(name), 1e-3)
    ge.march(5)
    oe.march(5)
    assert set(ge.kernel_forms.values()) == {'f3' if ge.ndim == 2 else 'f2'}
    assert ge.exact_passes == 0
    pair.same_euler(ge, oe)
    c = ge.ngstcell + ge.ncell // 2
    for a, i, v in (('so0n', (c, 0), 1e15), ('so0n', (c, ge.ndim + 1), 1e16),
                    ('so1n', (c - 1, 1, 0), np.inf)):
        getattr(ge, a).ndarray[i] = v
        getattr(oe, a)[i] = v
    ge.march(2)
    oe.march(2)
    assert ge.exact_passes > 0
    for t in ('so0n', 'so1n', 'cflo', 'cflc', 'so0t'):
        assert np.array_equal(getattr(ge, t).ndarray, getattr(oe, t),
                              equal_nan=True), t


@pytest.mark.parametrize('m', [134, 135])
def test_lane_limit(orc, monkeypatch, m):
    # 35912 triangles take it, 36450 are timed; either equals the oracle.
    from solvcon_amd.gen import tri_mesh_def
    print('case: lane limit', m, flush=True)
    monkeypatch.delenv('SC_EULER_FORM', raising=False)
    ge, oe = _pair(orc, tri_mesh_def(m, seed=4), 1e-4)
    ge.march(3)
    oe.march(3)
    if m == 134:
        assert ge.kernel_forms == {4: 'f3'}
    pair.same_euler(ge, oe)


# Untimed up to the limit of each type, timed beyond (the eight-lane types' lies
# far below the tetrahedra's); either equals the oracle.
@pytest.mark.parametrize('kind,n,timed', [
    ('prism', 28, False), ('prism', 29, True), ('hex', 41, False),
    ('hex', 42, True), ('tet', 21, False), ('quad', 189, False),
    ('quad', 190, True), ('all', 30, True)])
def test_lane_limit_by_type(orc, monkeypatch, capfd, kind, n, timed):
    from solvcon_amd.gen import mixed_mesh_def, rect_mesh_def
    print('case: lane limit', kind, n, flush=True)
    monkeypatch.delenv('SC_EULER_FORM', raising=False)
    monkeypatch.setenv('SC_EULER_TUNE_LOG', '1')
    if kind == 'quad':
        defn = rect_mesh_def(n, n, kind='quad', seed=3, jitter=0.2)
    else:
        frac = {'prism': (0.0, 1.0), 'hex': (0.0, 0.0),
                'tet': ((n + 1.0) / n, 0.0), 'all': (0.1, 0.85)}[kind]
        defn = mixed_mesh_def(n, seed=3, tet_frac=frac[0], prism_frac=frac[1])
    ge, oe = _pair(orc, defn, 1e-4)
    ge.march(2)
    assert ('EulerCore tuning' in capfd.readouterr().err) == timed
    if not timed:
        assert set(ge.kernel_forms.values()) == {'f3' if ge.ndim == 2 else 'f2'}
    oe.march(2)
    pair.same_euler(ge, oe)


@pytest.mark.parametrize('name,waves', [('tri-64x64', 512), ('mixed-7', 98)])
def test_lane_exact_only(orc, monkeypatch, name, waves):
    # A state out of range everywhere: the wavefronts of the first launch that
    # meet it run both forms, the launches after it the exact form alone
    # (counted once per group), until the next march.
    print('case: lane exact only', name, flush=True)
    monkeypatch.delenv('SC_EULER_FORM', raising=False)
    ge, oe = _pair(orc, _defn(name), 1e-3)
    steps = 10
    ge.march(steps)
    oe.march(steps)
    assert ge.exact_passes == 0
    for a, x in ((ge.so0n.ndarray, ge.ngstcell), (oe.so0n, oe.ngstcell)):
        a[x:, 0] *= 1e15
        a[x:, -1] *= 1e16
    ge.march(steps)
    oe.march(steps)
    groups = len(ge.kernel_forms)
    assert 0 < ge.exact_passes <= waves + 2 * steps * groups
    pair.same_euler(ge, oe)
    before = ge.exact_passes
    ge.march(1)
    assert ge.exact_passes > before


@pytest.mark.parametrize('n,form', [(189, 'f3'), (191, 'f1')])
def test_no_prefetch_falls_back(orc, monkeypatch, n, form):
    # Quadrilaterals have no three-wave geometry prefetch: what runs in its
    # place is the face lanes only up to their limit (36000 cells).
    from solvcon_amd.gen import rect_mesh_def
    print('case: no prefetch', n, flush=True)
    monkeypatch.setenv('SC_EULER_FORM', 'f3g')
    ge, oe = _pair(orc, rect_mesh_def(n, n, kind='quad', seed=3, jitter=0.2),
                   1e-4)
    ge.march(2)
    oe.march(2)
    assert ge.kernel_forms == {3: form}
    pair.same_euler(ge, oe)
