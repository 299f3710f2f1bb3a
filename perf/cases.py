"""The work that users of solvcon_amd have it do, as measurable cases.

A case is one of these, each through the package's public classes:

tube        a 1D shock tube (``Euler1DCore``): load the initial state, set up
            the march, run ``march_alpha1`` or ``march_alpha2``, read so0 and
            so1.  From the few hundred points of a teaching plot through the
            2001-point Sod tube of bench.py to half a million points.
scalar      a periodic 1D scalar march (``LinearScalarSolver``,
            ``InviscidBurgersSolver``).
reflection  the oblique-shock reflection session: an ``EulerCore`` with two
            inlets, a slip wall and a non-reflective edge on a rectangle of
            quadrilaterals or triangles goes on marching and its state is
            read, as the obsrefl application does between its plots.
riemann     one 2D solve on a solver in hand: load a four-quadrant Riemann
            box on a jittered triangle mesh, apply the boundaries, march,
            read so0n and so1n.  The largest is bench.py's 2D workload.
blast       the same in 3D: a spherical blast on the mixed hexahedron /
            tetrahedron / prism / pyramid block, slip walls on three sides.
setup       everything before the first step of a solve: mesh build
            (interior, boundary, ghosts), solver construction with its CE
            geometry, initial state, boundaries and the CFL time step.
batch       many small independent 2D solves in one ``BatchedEuler`` march,
            sizes and step counts drawn as ``batch_config`` draws them.

Sizes come from bench.py, batch_config, the request mix of serve.py
(1e3 to 2e6 cells, 100 to 1000 steps) and the tests (64 x 16 boxes).
"""

import math

import numpy as np
import torch

import solvcon_amd as sc
from solvcon_amd import batch as sb
from solvcon_amd import gen
from solvcon_amd import spacetime as st

GAMMA = 1.4


def listed():
    return [
        # The smallest: a tube with a few hundred points, as plotted live.
        {'name': 'tube-small', 'kind': 'tube', 'n': 201, 'steps': 60,
         'alpha': 2},
        # The Sod tube of bench.py --config 1d.
        {'name': 'tube-sod', 'kind': 'tube', 'n': 2001, 'steps': 600,
         'alpha': 2},
        # A finely resolved tube: throughput, not latency.
        {'name': 'tube-large', 'kind': 'tube', 'n': 500001, 'steps': 100,
         'alpha': 2},
        # A scalar march of ordinary size.
        {'name': 'burgers', 'kind': 'scalar', 'eq': 'burgers', 'n': 1000,
         'steps': 500, 'alpha': 2},
        # The obsrefl application's default 64 x 16 boxes, quadrilaterals.
        {'name': 'reflection-quad', 'kind': 'reflection', 'cell': 'quad',
         'nx': 64, 'ny': 16, 'steps': 50},
        # A 2D solve of the size most batched and served requests have.
        {'name': 'riemann-medium', 'kind': 'riemann', 'm': 96, 'steps': 100},
        # bench.py --config 2d: 2,097,152 triangles, 500 steps.
        {'name': 'riemann-large', 'kind': 'riemann', 'm': 1024,
         'steps': 500},
        # A coarse 3D solve (odd size), launch and latency bound.
        {'name': 'blast-small', 'kind': 'blast', 'n': 15, 'steps': 100},
        # A 3D solve far beyond the caches.
        {'name': 'blast-large', 'kind': 'blast', 'n': 80, 'steps': 200},
        # Set-up of a 2D and of a 3D solve.
        {'name': 'setup-tri', 'kind': 'setup', 'cell': 'tri', 'm': 256},
        {'name': 'setup-block', 'kind': 'setup', 'cell': 'block', 'm': 40},
        # 48 instances of the batched workload's distribution.
        {'name': 'batch-tri', 'kind': 'batch', 'ninst': 48, 'lo': 1000,
         'hi': 200000, 'smin': 100, 'smax': 1000},
    ]


def draw(rng):
    def logu(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(['tube', 'tube', 'scalar', 'reflection', 'riemann',
                       'riemann', 'blast', 'blast', 'setup', 'batch'])
    if kind == 'tube':
        n = logu(100, 250000) * 2 + 1
        return {'kind': kind, 'n': n, 'alpha': rng.choice([1, 2, 2]),
                'steps': min(logu(20, 600), max(20, 50000000 // n))}
    if kind == 'scalar':
        n = logu(32, 50000)
        return {'kind': kind, 'eq': rng.choice(['linear', 'burgers']),
                'n': n, 'alpha': rng.choice([0, 1, 2]),
                'steps': min(logu(50, 1000), max(50, 20000000 // n))}
    if kind == 'reflection':
        ny = logu(4, 128)
        return {'kind': kind, 'cell': rng.choice(['quad', 'tri']),
                'nx': 4 * ny + rng.randrange(4), 'ny': ny,
                'steps': logu(20, 100)}
    if kind == 'riemann':
        m = logu(16, 1000)
        return {'kind': kind, 'm': m,
                'steps': min(logu(20, 500), max(20, 500000000 // (m * m)))}
    if kind == 'blast':
        n = logu(6, 78)
        return {'kind': kind, 'n': n,
                'steps': min(logu(20, 200),
                             max(20, 100000000 // (n * n * n)))}
    if kind == 'setup':
        if rng.random() < 0.5:
            return {'kind': kind, 'cell': 'tri', 'm': logu(16, 500)}
        return {'kind': kind, 'cell': 'block', 'm': logu(6, 48)}
    return {'kind': kind, 'ninst': rng.randrange(8, 49), 'lo': 1000,
            'hi': logu(4000, 200000), 'smin': 100,
            'smax': rng.randrange(120, 900)}


# ------------------------------------------------------------------------
# What a user's program holds before the call.
# ------------------------------------------------------------------------

def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _tube_input(case, seed):
    """Grid, primitive states and dt of a shock tube: Sod's pressure and
    density ratios varied by the seed, the largest CFL number about 0.75."""
    r = _rng(seed)
    n = case['n']
    x = np.linspace(-1.0, 1.0, n)
    left = (1.0 + 0.2 * r.uniform(), 0.0, 1.0 + 0.2 * r.uniform())
    right = (0.125 + 0.05 * r.uniform(), 0.0, 0.1 + 0.05 * r.uniform())
    prim = np.where((x < 0.0)[:, None], np.array(left), np.array(right))
    rho, u, p = prim.T
    so0 = np.stack([rho, rho * u, p / (GAMMA - 1.0) + 0.5 * rho * u * u],
                   axis=1)
    return x, so0, 0.4 / 600 * 2000 / (n - 1)


def _scalar_input(case, seed):
    """Grid size, dt and initial sine of a periodic scalar march at CFL
    0.4 to 0.9."""
    r = _rng(seed)
    n = case['n']
    dt = (0.4 + 0.5 * r.uniform()) * 2.0 * math.pi / n
    shift, amp = r.uniform(), 0.5 + 0.5 * r.uniform()
    return n, dt, shift, amp


def _oblique(mach, theta, rho, p):
    """State behind the weak oblique shock that turns a Mach ``mach``
    stream along +x by -theta: (rho, u, v, p)."""
    def turn(b):
        s2 = (mach * math.sin(b)) ** 2
        return math.atan(2.0 / math.tan(b) * (s2 - 1.0)
                         / (mach * mach * (GAMMA + math.cos(2 * b)) + 2.0))
    lo, hi = math.asin(1.0 / mach), math.radians(60.0)
    for _ in range(200):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if turn(mid) < theta else (lo, mid)
    b = 0.5 * (lo + hi)
    m2 = (mach * math.sin(b)) ** 2
    pr = 1.0 + 2.0 * GAMMA / (GAMMA + 1.0) * (m2 - 1.0)
    rr = (GAMMA + 1.0) * m2 / ((GAMMA - 1.0) * m2 + 2.0)
    mn = math.sqrt((1.0 + 0.5 * (GAMMA - 1.0) * m2)
                   / (GAMMA * m2 - 0.5 * (GAMMA - 1.0)))
    a = math.sqrt(GAMMA * p * pr / (rho * rr))
    v = mn / math.sin(b - theta) * a
    return rho * rr, v * math.cos(theta), -v * math.sin(theta), p * pr


EXTENT = (4.0, 1.0)


def _reflection_input(case, seed):
    r = _rng(seed)
    mach = 2.8 + 0.4 * r.uniform()
    theta = math.radians(9.0 + 2.0 * r.uniform())
    rho, p = 1.0, 1.0 / GAMMA
    u = mach
    two = _oblique(mach, theta, rho, p)
    defn = gen.rect_mesh_def(case['nx'], case['ny'], extent=EXTENT,
                             kind=case['cell'], seed=seed % 1000)
    return defn, (rho, u, 0.0, p), two


def _mesh_input(case, seed):
    """(mesh definition, state function of the centroids, CFL number) of a
    riemann, blast or setup case."""
    two_d = case['kind'] == 'riemann' or case.get('cell') == 'tri'
    if two_d:
        defn = gen.tri_mesh_def(case['m'], seed=seed)
        rho, p = gen.riemann_box(seed)
        return (defn, lambda c: gen.quadrant_state(c, rho, p, GAMMA), 0.8)
    n = case['n'] if case['kind'] == 'blast' else case['m']
    defn = gen.mixed_mesh_def(n, seed=seed)
    p_in = 8.0 + 4.0 * _rng(seed).uniform()
    # The blast spans at least three cells (the request mix does the same).
    return (defn, lambda c: gen.blast_state(c, GAMMA, r=max(0.1, 3.0 / n),
                                            p_in=p_in), 0.6)


def _batch_sizes(case):
    """Boxes per side and step counts of a batch, as batch_config draws
    them; they belong to the case, meshes and states come from the seed."""
    m, _, _, steps = sb.batch_config(
        case['ninst'], seed=case['ninst'], lo=float(case['lo']),
        hi=float(case['hi']), smin=case['smin'], smax=case['smax'])
    return m, steps


def _boundaries(mesh, two_d):
    """Slip walls on x = 0, y = 0, z = 0 of a block, non-reflective faces
    elsewhere; all non-reflective in 2D."""
    bf = mesh.bndfcs.ndarray[:, 0].copy()
    if two_d:
        return [('nonrefl', bf)]
    c = mesh.fccnd.ndarray[mesh.ngstface + bf]
    wall = (np.abs(c) < 1e-12).any(axis=1)
    return [('slipwall', bf[wall]), ('nonrefl', bf[~wall])]


def _build(defn):
    ndim, ndcrd, cltpn, clnds = defn
    mesh = sc.StaticMesh(ndim=ndim, nnode=ndcrd.shape[0], nface=0,
                         ncell=cltpn.shape[0])
    mesh.ndcrd.ndarray[...] = ndcrd
    mesh.cltpn.ndarray[...] = cltpn
    mesh.clnds.ndarray[:, :clnds.shape[1]] = clnds
    mesh.build_interior(do_metric=True, build_edge=False)
    mesh.build_boundary()
    mesh.build_ghost()
    return mesh


def _ready(mesh, state_of, cfl):
    """An EulerCore with its initial state, boundaries and CFL time step;
    also the initial body rows."""
    two_d = mesh.ndim == 2
    g = mesh.ngstcell
    core = sc.EulerCore(mesh=mesh, time_increment=1.0)
    core.init_solution(GAMMA, 1.0, [0.0] * mesh.ndim, 1.0)
    body = state_of(mesh.clcnd.ndarray[g:])
    core.so0n.ndarray[g:] = body
    for kind, faces in _boundaries(mesh, two_d):
        getattr(core, 'add_' + kind)(faces)
    core.bc_soln()
    core.bc_dsoln()
    dt = core.cfl_dt(cfl)
    core.set_time_increment(dt)
    return core, body, dt


def prepare(case, seed):
    kind = case['kind']
    if kind == 'tube':
        x, so0, dt = _tube_input(case, seed)
        core = sc.onedim.Euler1DCore(ncoord=case['n'], time_increment=dt)
        core.coord[...] = x
        core.gamma.fill(GAMMA)
        return {'kind': kind, 'core': core, 'so0': so0, 'case': case}
    if kind == 'scalar':
        n, dt, shift, amp = _scalar_input(case, seed)
        grid = st.Grid(0.0, 2.0 * math.pi, n)
        cls = (st.LinearScalarSolver if case['eq'] == 'linear'
               else st.InviscidBurgersSolver)
        x = np.array(grid.xcoord)
        return {'kind': kind, 'case': case,
                'core': cls(grid=grid, time_increment=dt),
                'u0': amp * np.sin(x - shift), 'u1': amp * np.cos(x - shift)}
    if kind == 'reflection':
        defn, one, two = _reflection_input(case, seed)
        mesh = _build(defn)
        core = sc.EulerCore(mesh=mesh, time_increment=1.0)
        core.init_solution(GAMMA, one[0], list(one[1:3]), one[3])
        left, top, bottom, right = gen.edge_faces(
            mesh.bndfcs.ndarray[:, 0], mesh.fccnd.ndarray[mesh.ngstface:],
            EXTENT)
        core.add_inlet(left, list(one) + [GAMMA])
        core.add_inlet(top, list(two) + [GAMMA])
        core.add_slipwall(bottom)
        core.add_nonrefl(right)
        core.bc_soln()
        core.bc_dsoln()
        core.set_time_increment(core.cfl_dt(0.45))
        return {'kind': kind, 'mesh': mesh, 'core': core, 'case': case,
                'g': mesh.ngstcell}
    if kind in ('riemann', 'blast'):
        defn, state_of, cfl = _mesh_input(case, seed)
        mesh = _build(defn)
        core, body, _ = _ready(mesh, state_of, cfl)
        return {'kind': kind, 'mesh': mesh, 'core': core, 'body': body,
                'case': case, 'g': mesh.ngstcell}
    if kind == 'setup':
        defn, state_of, cfl = _mesh_input(case, seed)
        return {'kind': kind, 'defn': defn, 'state': state_of, 'cfl': cfl,
                'case': case}
    m, steps = _batch_sizes(case)
    mseed, rseed = _rng(seed).integers(0, 2 ** 31, (2, case['ninst']))
    state_of = sb.config_states(rseed, GAMMA)
    b = sb.BatchedEuler(sb.config_defs(m, mseed), state_of, steps,
                        gamma=GAMMA)
    cen = b.mesh.clcnd.ndarray[b.ngst:]
    body = np.concatenate([state_of(cen[b.coff[k]:b.coff[k + 1]], k)
                           for k in range(b.ninst)])
    return {'kind': kind, 'batch': b, 'core': b.core, 'body': body,
            'g': b.ngst, 'case': case}


# ------------------------------------------------------------------------
# One pass.
# ------------------------------------------------------------------------

def _load(core, body, g):
    core.so0n.ndarray[g:] = body
    core.so1n.ndarray[...] = 0.0
    core.bc_soln()
    core.bc_dsoln()


def run(s):
    kind, case = s['kind'], s['case']
    if kind == 'setup':
        mesh = _build(s['defn'])
        g = mesh.ngstcell
        core, _, dt = _ready(mesh, s['state'], s['cfl'])
        return {'clfcs': mesh.clfcs.ndarray[g:],
                'fccls': mesh.fccls.ndarray[mesh.ngstface:],
                'clvol': mesh.clvol.ndarray[g:],
                'clcnd': mesh.clcnd.ndarray[g:],
                'cevol': core.cevol.ndarray[g:],
                'cecnd': core.cecnd.ndarray[g:], 'dt': dt}
    core = s['core']
    if kind == 'tube':
        core.so0[...] = s['so0']
        core.so1[...] = 0.0
        core.setup_march()
        if case['alpha'] == 1:
            core.march_alpha1(case['steps'])
        else:
            core.march_alpha2(case['steps'])
        return {'so0': core.so0, 'so1': core.so1}
    if kind == 'scalar':
        core.so0.ndarray[:, 0] = s['u0']
        core.so1.ndarray[:, 0] = s['u1']
        core.setup_march()
        getattr(core, 'march_alpha%d' % case['alpha'])(case['steps'])
        return {'so0': core.so0.ndarray, 'so1': core.so1.ndarray}
    if kind == 'batch':
        _load(core, s['body'], s['g'])
        s['batch'].march()
    elif kind == 'reflection':
        core.march(case['steps'])
    else:
        _load(core, s['body'], s['g'])
        core.march(case['steps'])
    g = s['g']
    return {'so0n': core.so0n.ndarray[g:], 'so1n': core.so1n.ndarray[g:]}


# ------------------------------------------------------------------------
# What a pass cannot do without.
# ------------------------------------------------------------------------

# Cell type: (dimensions, faces, sub-faces, gradient elements).
SHAPE = {3: (2, 4, 8, 4), 4: (2, 3, 6, 3), 5: (3, 6, 24, 8), 6: (3, 4, 12, 4),
         7: (3, 5, 18, 6), 8: (3, 5, 16, 6)}
CACHE = 256e6  # last-level cache: tables that fit stay on the chip


def _substep(t):
    """(geometry bytes, state bytes read, state bytes written, operations) of
    one cell of type t in one substep: the CE volumes, centroids, sub-face
    centroids and normals and the neighbour list; so0, so1, gamma in; so0,
    so1 and two CFL numbers out.  A division or square root counts as one."""
    d, f, s, e = SHAPE[t]
    q = d + 2
    geo = 8 * (f + 1) + 8 * d * (f + 1) + 16 * s * d + 4 * f
    read = 8 * (q + q * d + 1)
    wrote = 8 * (q + q * d + 2)
    face = q * (3 * d + 2) + 12 * q + 2 * q * q * d
    sub = q * (3 * d + 1) + q * (d * (2 * q + 2) + 2)
    grad = f * (6 * d + q * (2 * d + 2)) + e * 12 * d
    eq = e * (2 * d * d + 6 * d + 8) + 4
    return geo, read, wrote, f * face + s * sub + grad + q * eq + 30


def _mix(case):
    """Cells by type."""
    kind = case['kind']
    if kind == 'riemann' or case.get('cell') == 'tri' and kind == 'setup':
        return {4: 2 * case['m'] ** 2}
    if kind == 'reflection':
        n = case['nx'] * case['ny']
        return {3: n} if case['cell'] == 'quad' else {4: 2 * n}
    n = case['n'] if kind == 'blast' else case['m']
    kp = int(round(0.2 * n))
    kt = max(int(round(0.3 * n)) - 1, 0)
    tr = 1 if kt > 0 else 0
    a = n * n
    return {5: a * (n - kp - kt - tr), 6: a * (5 * kt + 2 * tr),
            7: 2 * a * kp, 8: 5 * a * tr}


def _march_work(mix, steps):
    geo, read, wrote, ops = (sum(c * _substep(t)[k] for t, c in mix.items())
                             for k in range(4))
    if geo + read + wrote > CACHE:
        return 2 * steps * (geo + read + wrote), 2 * steps * ops
    return geo + read + wrote, 2 * steps * ops


def work(case):
    kind = case['kind']
    if kind == 'tube':
        n, steps = case['n'], case['steps']
        # Per new point: two elements' shared fluxes and one gradient.
        return {'bytes': 14 * 8 * n, 'flops': n * steps * 240}
    if kind == 'scalar':
        n, steps = 2 * case['n'], case['steps']
        return {'bytes': 5 * 8 * n, 'flops': n * steps * 50}
    if kind == 'batch':
        m, steps = _batch_sizes(case)
        b = f = 0
        geo, read, wrote, ops = _substep(4)
        fits = (geo + read + wrote) * float((2 * m * m).sum()) <= CACHE
        for mk, sk in zip(m, steps):
            n = 2 * int(mk) ** 2
            b += n * (geo + read + wrote) * (1 if fits else 2 * int(sk))
            f += n * ops * 2 * int(sk)
        return {'bytes': b, 'flops': f}
    mix = _mix(case)
    if kind == 'setup':
        # Nodes and cell nodes in; the mesh tables and the CE geometry out.
        b = f = 0
        for t, c in mix.items():
            d, nf, s, _ = SHAPE[t]
            nn = {3: 4, 4: 3, 5: 8, 6: 4, 7: 6, 8: 5}[t]
            b += c * (4 * (nn + 1) + 8 * d + 28 + 8 * (d + 1)
                      + nf * (8 * d + 10 + 8) + _substep(t)[0])
            f += c * s * 60 * d
        return {'bytes': b, 'flops': f}
    b, f = _march_work(mix, case['steps'])
    return {'bytes': b, 'flops': f}


def tolerance(case):
    """All arithmetic is FP64; the values are about four times the distance
    to exact() or more.  The 2D Riemann marches amplify the last bits where
    the limiter switches: 1e-13 in 10 steps, 1e-3 in the gradients in 100.
    The reflection starts from a uniform stream, whose gradients are
    rounding noise that the limiter's weights divide by."""
    kind = case['kind']
    if kind == 'setup':
        return {'rel': 2e-13}
    if kind in ('tube', 'scalar'):
        return {'rel': 1e-10}
    if kind == 'blast':
        return {'rel': 1e-9}
    if kind == 'reflection':
        return {'rel': 1e-6}
    return {'rel': 5e-3}


# ------------------------------------------------------------------------
# The same results from plain torch in 64 bits.
# ------------------------------------------------------------------------

def exact(case, seed):
    kind = case['kind']
    dev = 'cuda' if torch.cuda.is_available() else 'cpu'
    if kind == 'tube':
        # Kernel launches of about 10 us each; 250 of them per step.
        if case['n'] * case['steps'] > 5e7:
            return None
        return _exact_tube(case, seed, dev)
    if kind == 'scalar':
        if case['n'] * case['steps'] > 5e7:
            return None
        return _exact_scalar(case, seed, dev)
    if kind == 'setup':
        defn, _, cfl = _mesh_input(case, seed)
        m = _Mesh64(defn, dev)
        _, state_of, _ = _mesh_input(case, seed)
        body = torch.as_tensor(state_of(m.clcnd.cpu().numpy()), device=dev)
        vol, cen = m.ce_tables()
        return {'clfcs': None, 'fccls': None, 'clvol': m.clvol.cpu().numpy(),
                'clcnd': m.clcnd.cpu().numpy(), 'cevol': vol.cpu().numpy(),
                'cecnd': cen.cpu().numpy(), 'dt': m.cfl_dt(body, cfl)}
    if kind == 'batch':
        return None  # every instance would be a march of its own
    cells = sum(_mix(case).values())
    if case['steps'] > 100 or cells * case['steps'] > 4e6:
        return None
    if kind == 'reflection':
        defn, one, two = _reflection_input(case, seed)
        m = _Mesh64(defn, dev)
        c = m.gface
        edge = (c[:, 0].abs() < 1e-9, (c[:, 1] - EXTENT[1]).abs() < 1e-9,
                c[:, 1].abs() < 1e-9, (c[:, 0] - EXTENT[0]).abs() < 1e-9)
        body = torch.tensor([one[0], one[0] * one[1], one[0] * one[2],
                             one[3] / (GAMMA - 1.0) + 0.5 * one[0]
                             * (one[1] ** 2 + one[2] ** 2)],
                            dtype=torch.float64, device=dev)
        body = body.expand(m.N, 4).clone()
        bc = [('inlet', edge[0], one), ('inlet', edge[1], two),
              ('slipwall', edge[2], None), ('nonrefl', edge[3], None)]
        cfl = 0.45
    else:
        defn, state_of, cfl = _mesh_input(case, seed)
        m = _Mesh64(defn, dev)
        body = torch.as_tensor(state_of(m.clcnd.cpu().numpy()), device=dev)
        wall = (m.gface.abs() < 1e-12).any(1) & (m.nd == 3)
        bc = [('slipwall', wall, None), ('nonrefl', ~wall, None)]
    s0, s1 = m.march(body, bc, m.cfl_dt(body, cfl), case['steps'])
    return {'so0n': s0.cpu().numpy(), 'so1n': s1.cpu().numpy()}


def _exact_tube(case, seed, dev):
    x, so0, dt = _tube_input(case, seed)
    n = case['n']
    x = torch.as_tensor(x, device=dev)
    s0 = torch.as_tensor(so0, device=dev).clone()
    s1 = torch.zeros_like(s0)
    h, q = dt / 2.0, dt / 4.0
    ga = GAMMA

    def boundary():
        for a in (s0, s1):
            a[1] = a[2]
            a[n - 2] = a[n - 3]

    def half(odd):
        first = 1 if odd else 2
        c = torch.arange(first, n - first, 2, device=dev)
        xm, xc, xp = x[c - 1], x[c], x[c + 1]
        u, ux = s0[c], s1[c]
        r, m, e = u.T
        one = torch.ones_like(r)
        v = m / r
        zero = torch.zeros_like(r)
        jac = torch.stack([
            zero, one, zero,
            0.5 * (ga - 3) * v * v, (3 - ga) * v, (ga - 1) * one,
            (ga - 1) * v ** 3 - ga * v * e / r,
            ga * e / r - 1.5 * (ga - 1) * v * v, ga * v], 1).view(-1, 3, 3)
        f = torch.stack([m, (ga - 1) * e + 0.5 * (3 - ga) * m * v,
                         ga * v * e - 0.5 * (ga - 1) * m * v * v], 1)
        ut = -(jac @ ux[:, :, None])[:, :, 0]
        ft = (jac @ ut[:, :, None])[:, :, 0]
        ctr = 0.5 * (xm + xp)
        up = u + (xc - ctr)[:, None] * ux + h * ut
        dl, dr = (xp - xc)[:, None], (xc - xm)[:, None]
        off = (xc - ctr)[:, None]
        tl = h * (f - off * ut + q * ft)
        right = dl * (u + (0.5 * (xc + xp) - ctr)[:, None] * ux) + tl
        left = dr * (u + (0.5 * (xc + xm) - ctr)[:, None] * ux) - tl
        new = (right[:-1] + left[1:]) / (xc[1:] - xc[:-1])[:, None]
        gn = (new - up[:-1]) / dl[:-1]
        gp = (up[1:] - new) / dr[1:]
        a = case['alpha']
        fn, fp = gn.abs() ** a, gp.abs() ** a
        s0[c[:-1] + 1] = new
        s1[c[:-1] + 1] = (fp * gn + fn * gp) / (fp + fn + 1e-100)

    for _ in range(case['steps']):
        half(False)
        boundary()
        half(True)
    return {'so0': s0.cpu().numpy(), 'so1': s1.cpu().numpy()}


def _exact_scalar(case, seed, dev):
    n, dt, shift, amp = _scalar_input(case, seed)
    h = 0.5 * (2.0 * math.pi / n)
    # Two points beyond each end; solution elements at even offsets from 2.
    x = (torch.arange(2 * n + 5, dtype=torch.float64, device=dev) - 2) * h
    s0 = amp * torch.sin(x - shift)
    s1 = amp * torch.cos(x - shift)
    hd, qd = 0.5 * dt, 0.25 * dt
    linear = case['eq'] == 'linear'
    a = case['alpha']

    def half(odd):
        X = torch.arange(2 if odd else 3, 2 * n + 3, 2, device=dev)
        if not odd:
            X = X[:n]
        l, r = X - 1, X + 1
        u, ux = s0, s1
        # An element's own cell is symmetric on a uniform grid.
        t = (u + 0.0 * ux if linear else 0.5 * u * u)
        flux = hd * (t - qd * (ux if linear else u * u * ux))
        new = ((h * (u + 0.5 * h * ux))[l] + flux[l]
               + (h * (u - 0.5 * h * ux))[r] - flux[r]) / (2.0 * h)
        up = u - hd * ux
        gn, gp = (new - up[l]) / h, (up[r] - new) / h
        fn, fp = gn.abs() ** a, gp.abs() ** a
        s0[X] = new
        s1[X] = (fp * gn + fn * gp) / (fp + fn + 2.2250738585072014e-308)
        if not odd:
            for b in (s0, s1):
                b[1] = b[2 * n + 1].clone()
                b[2 * n + 3] = b[3].clone()

    for _ in range(case['steps']):
        half(False)
        half(True)
    return {'so0': s0[:, None].cpu().numpy(), 'so1': s1[:, None].cpu().numpy()}


# Faces of each cell type as positions in its node list, and the faces that
# span each of its gradient elements.
FACES = {
    3: [(0, 1), (1, 2), (2, 3), (3, 0)],
    4: [(0, 1), (1, 2), (2, 0)],
    5: [(0, 3, 2, 1), (1, 2, 6, 5), (4, 5, 6, 7), (0, 4, 7, 3), (0, 1, 5, 4),
        (2, 3, 7, 6)],
    6: [(0, 2, 1), (0, 1, 3), (0, 3, 2), (1, 2, 3)],
    7: [(0, 1, 2), (3, 5, 4), (0, 3, 4, 1), (0, 2, 5, 3), (1, 4, 5, 2)],
    8: [(0, 4, 3), (1, 4, 0), (2, 4, 1), (3, 4, 2), (0, 3, 2, 1)],
}
SPANS = {
    3: [(0, 1), (1, 2), (2, 3), (3, 0)],
    4: [(0, 1), (1, 2), (2, 0)],
    5: [(1, 2, 4), (5, 2, 1), (3, 2, 5), (4, 2, 3), (4, 0, 1), (1, 0, 5),
        (5, 0, 3), (3, 0, 4)],
    6: [(2, 0, 1), (1, 0, 3), (3, 0, 2), (1, 3, 2)],
    7: [(4, 1, 3), (2, 1, 4), (3, 1, 2), (3, 0, 4), (4, 0, 2), (2, 0, 3)],
    8: [(0, 4, 1), (1, 4, 2), (2, 4, 3), (3, 4, 0), (0, 2, 3), (2, 0, 1)],
}


class _Mesh64(object):
    """A mesh definition's CE geometry and CESE march, vectorised over the
    cells of each type.  Rows are body cells in input order, then one ghost
    per boundary face."""

    def __init__(self, defn, dev):
        self.nd = nd = defn[0]
        xyz = torch.as_tensor(np.asarray(defn[1]), device=dev)
        tpn = np.asarray(defn[2])
        cln = np.asarray(defn[3]).astype(np.int64)
        self.N = N = len(tpn)
        self.dev = dev
        self.groups = []
        self.clcnd = torch.zeros(N, nd, dtype=torch.float64, device=dev)
        self.clvol = torch.zeros(N, dtype=torch.float64, device=dev)
        keys, where = [], []
        for t in sorted(set(tpn.tolist())):
            ids = torch.as_tensor(np.nonzero(tpn == t)[0], device=dev)
            fl = FACES[t]
            nn = max(max(f) for f in fl) + 1
            nodes = torch.as_tensor(cln[tpn == t][:, 1:1 + nn], device=dev)
            ctr = xyz[nodes].mean(1)
            fc, nml = [], []
            for j, f in enumerate(fl):
                ring = nodes[:, list(f)]
                p = xyz[ring]
                fc.append(self._face_centroid(p))
                nml.append(self._face_normal(p, fc[-1]))
                k = ring.sort(1).values
                key = k[:, 0]
                for c in range(1, nd):
                    key = key * xyz.shape[0] + k[:, c]
                keys.append(key)
                where.append(torch.stack([ids, torch.full_like(ids, j)], 1))
            fc = torch.stack(fc, 1)
            nml = torch.stack(nml, 1)
            du = ctr[:, None] - fc
            vob = (du * nml).sum(-1).abs()
            cen = ((fc + du / (nd + 1)) * vob[..., None]).sum(1) \
                / vob.sum(1, keepdim=True)
            out = ((fc - cen[:, None]) * nml).sum(-1)
            self.clcnd[ids] = cen
            self.clvol[ids] = out.abs().sum(1) / nd
            self.groups.append({'t': t, 'ids': ids, 'fc': fc, 'sgn':
                                torch.sign(out), 'nml': nml, 'xyz':
                                [xyz[nodes[:, list(f)]] for f in fl]})
        key, where = torch.cat(keys), torch.cat(where)
        order = torch.argsort(key, stable=True)
        ks = key[order]
        same = torch.zeros(len(ks) + 1, dtype=torch.bool, device=dev)
        same[1:-1] = ks[1:] == ks[:-1]
        first = same[1:]
        nbr = torch.full((N, 6), -1, dtype=torch.int64, device=dev)
        a = where[order[:-1][first[:-1]]]
        b = where[order[1:][first[:-1]]]
        nbr[a[:, 0], a[:, 1]] = b[:, 0]
        nbr[b[:, 0], b[:, 1]] = a[:, 0]
        lone = where[order[~(same[1:] | same[:-1])]]
        self.G = len(lone)
        self.gsrc = lone[:, 0]
        nbr[lone[:, 0], lone[:, 1]] = N + torch.arange(self.G, device=dev)
        self.gface = torch.zeros(self.G, nd, dtype=torch.float64, device=dev)
        self.gnml = torch.zeros_like(self.gface)
        for g in self.groups:
            g['nbr'] = nbr[g['ids']][:, :len(FACES[g['t']])]
            out = g['nbr'] >= N
            gi = g['nbr'][out] - N
            self.gface[gi] = g['fc'][out]
            n = g['nml'][out]
            self.gnml[gi] = n / n.norm(dim=1, keepdim=True)
        src = self.clcnd[self.gsrc]
        gcen = src + 2.0 * ((self.gface - src) * self.gnml).sum(
            1, keepdim=True) * self.gnml
        self.meshcen = torch.cat([self.clcnd, gcen])
        self.cen = self.meshcen.clone()
        for g in self.groups:
            self._ce(g)
            self.cen[g['ids']] = g['ccen']

    def _face_centroid(self, p):
        if self.nd == 2:
            return p.mean(1)
        c = p.mean(1, keepdim=True)
        nxt = p.roll(-1, 1)
        w = torch.linalg.cross(p - c, nxt - c).norm(dim=-1, keepdim=True)
        return ((c + p + nxt) / 3.0 * w).sum(1) / w.sum(1)

    def _face_normal(self, p, c):
        """Area times normal; its direction follows the node order."""
        if self.nd == 2:
            d = p[:, 1] - p[:, 0]
            return torch.stack([d[:, 1], -d[:, 0]], 1)
        r = p - c[:, None]
        return 0.5 * torch.linalg.cross(r, r.roll(-1, 1)).sum(1)

    def _ce(self, g):
        nd = self.nd
        mi = self.meshcen[g['ids']]
        vols, cens, sfc, sfn, s2f = [], [], [], [], []
        for j, p in enumerate(g['xyz']):
            me = self.meshcen[g['nbr'][:, j]]
            if nd == 2:
                a, b = p[:, 0], p[:, 1]

                def tri(c):
                    u, v = a - c, b - c
                    return u[:, 0] * v[:, 1] - u[:, 1] * v[:, 0]
                vi, ve = tri(mi).abs() / 2, tri(me).abs() / 2
                mom = (a + b + mi) / 3 * vi[:, None] \
                    + (a + b + me) / 3 * ve[:, None]
                vols.append(vi + ve)
                cens.append(mom)
                sg = torch.sign(tri(me))[:, None]
                for u, v in ((a, me), (me, b)):
                    d = v - u
                    sfc.append((u + v) / 2)
                    sfn.append(torch.stack([-d[:, 1], d[:, 0]], 1) * sg)
                    s2f.append(j)
                continue
            pf = g['fc'][:, j]
            sg = 0.5 * g['sgn'][:, j][:, None]
            vb, mom = 0.0, 0.0
            for k in range(p.shape[1]):
                a, b = p[:, k], p[:, (k + 1) % p.shape[1]]
                w = torch.linalg.cross(a - pf, b - pf)
                vi = (w * (mi - pf)).sum(1).abs() / 6
                ve = (w * (me - pf)).sum(1).abs() / 6
                vb = vb + vi + ve
                mom = mom + (a + b + pf + mi) / 4 * vi[:, None] \
                    + (a + b + pf + me) / 4 * ve[:, None]
                sfc.append((me + a + b) / 3)
                sfn.append(torch.linalg.cross(a - me, b - me) * sg)
                s2f.append(j)
            vols.append(vb)
            cens.append(mom)
        v = torch.stack(vols, 1)
        m = torch.stack(cens, 1)
        g['bvol'], g['bcen'] = v, m / v[..., None]
        g['cvol'] = v.sum(1)
        g['ccen'] = m.sum(1) / g['cvol'][:, None]
        g['sfc'], g['sfn'] = torch.stack(sfc, 1), torch.stack(sfn, 1)
        g['s2f'] = s2f
        g['dist'] = (g['bcen'] - g['ccen'][:, None]).norm(dim=-1).min(1).values

    def ce_tables(self):
        """The cevol and cecnd body rows: the cell's CE, then one basic CE
        per face."""
        vol = torch.zeros(self.N, 7, dtype=torch.float64, device=self.dev)
        cen = torch.zeros(self.N, 7, self.nd, dtype=torch.float64,
                          device=self.dev)
        for g in self.groups:
            k = g['bvol'].shape[1]
            vol[g['ids'], 0] = g['cvol']
            vol[g['ids'], 1:k + 1] = g['bvol']
            cen[g['ids'], 0] = g['ccen']
            cen[g['ids'], 1:k + 1] = g['bcen']
        return vol, cen.reshape(self.N, -1)

    def _wave(self, u):
        ke = (u[:, 1:-1] ** 2).sum(1) / (2 * u[:, 0])
        p = ((GAMMA - 1) * (u[:, -1] - ke)).clamp(min=0.0)
        return torch.sqrt(GAMMA * p / u[:, 0]) \
            + (u[:, 1:-1] ** 2).sum(1).sqrt() / u[:, 0], p, ke

    def cfl_dt(self, body, cfl):
        worst = 0.0
        for g in self.groups:
            w = self._wave(body[g['ids']])[0]
            worst = max(worst, float((0.5 * w / g['dist']).max()))
        return cfl / worst

    def _jac(self, u):
        """Flux F[r, k, d] and Jacobian J[r, k, m, d] of rows u[r, q]."""
        nd, q = self.nd, self.nd + 2
        ga = GAMMA
        v = u[:, 1:-1] / u[:, :1]
        e = u[:, -1] / u[:, 0]
        v2 = (v * v).sum(1)
        p = (ga - 1) * (u[:, -1] - 0.5 * u[:, 0] * v2)
        F = torch.zeros(len(u), q, nd, dtype=u.dtype, device=u.device)
        J = torch.zeros(len(u), q, q, nd, dtype=u.dtype, device=u.device)
        for d in range(nd):
            F[:, 0, d] = u[:, 1 + d]
            F[:, -1, d] = (u[:, -1] + p) * v[:, d]
            J[:, 0, 1 + d, d] = 1.0
            for k in range(nd):
                F[:, 1 + k, d] = u[:, 1 + k] * v[:, d]
                J[:, 1 + k, 0, d] = -v[:, k] * v[:, d]
                J[:, 1 + k, 1 + k, d] += v[:, d]
                J[:, 1 + k, 1 + d, d] += v[:, k]
                J[:, -1, 1 + k, d] = -(ga - 1) * v[:, k] * v[:, d]
            F[:, 1 + d, d] += p
            J[:, 1 + d, 0, d] += 0.5 * (ga - 1) * v2
            J[:, 1 + d, 1:1 + nd, d] -= (ga - 1) * v
            J[:, 1 + d, -1, d] = ga - 1
            J[:, -1, 0, d] = ((ga - 1) * v2 - ga * e) * v[:, d]
            J[:, -1, 1 + d, d] += ga * e - 0.5 * (ga - 1) * v2
            J[:, -1, -1, d] = ga * v[:, d]
        return F, J

    def _ghost0(self, bc, u):
        out = u[self.gsrc].clone()
        n = self.gnml
        for kind, at, val in bc:
            if kind == 'slipwall':
                mom = out[at][:, 1:-1]
                nn = n[at]
                out[at, 1:-1] = mom - 2 * (mom * nn).sum(1, True) * nn
            elif kind == 'inlet':
                r, v, p = val[0], val[1:-1], val[-1]
                out[at] = torch.tensor(
                    [r] + [r * c for c in v]
                    + [p / (GAMMA - 1) + 0.5 * r * sum(c * c for c in v)],
                    dtype=u.dtype, device=u.device)
        return out

    def _ghost1(self, bc, ux):
        out = ux[self.gsrc].clone()
        n = self.gnml
        for kind, at, _ in bc:
            g, nn = out[at], n[at]
            if kind == 'inlet':
                out[at] = 0.0
                continue
            along = torch.einsum('rkd,rd->rk', g, nn)[..., None] \
                * nn[:, None]
            if kind == 'nonrefl':
                out[at] = g - along
                continue
            g = g - 2 * along
            mom = g[:, 1:-1]
            g[:, 1:-1] = mom - 2 * nn[..., None] * torch.einsum(
                'rk,rkd->rd', nn, mom)[:, None]
            out[at] = g
        return out

    def march(self, body, bc, dt, steps, sigma0=3.0, taumin=0.0,
              tauscale=1.0):
        nd, q = self.nd, self.nd + 2
        h, qt = dt * 0.5, dt * 0.25
        s0 = torch.cat([body, self._ghost0(bc, body)])
        s1 = torch.zeros(len(s0), q, nd, dtype=s0.dtype, device=s0.device)
        for _ in range(2 * steps):
            F, J = self._jac(s0)
            ut = -torch.einsum('rkmd,rmd->rk', J, s1)
            pre = torch.empty(self.N, q, dtype=s0.dtype, device=s0.device)
            new = torch.empty_like(pre)
            grad = torch.empty(self.N, q, nd, dtype=s0.dtype,
                               device=s0.device)
            for g in self.groups:
                ids, j, s2f = g['ids'], g['nbr'], g['s2f']
                js, j1, cj = s0[j], s1[j], self.cen[j]
                tot = ((js + torch.einsum('nfd,nfkd->nfk', g['bcen'] - cj,
                                          j1)) * g['bvol'][..., None]).sum(1)
                du = qt * ut[j][:, s2f] + torch.einsum(
                    'nsd,nskd->nsk', g['sfc'] - cj[:, s2f], j1[:, s2f])
                flux = F[j][:, s2f] + torch.einsum('nskmd,nsm->nskd',
                                                   J[j][:, s2f], du)
                tot = tot - h * torch.einsum('nskd,nsd->nk', flux, g['sfn'])
                u = tot / g['cvol'][:, None]
                pre[ids] = u
                w, p, ke = self._wave(u)
                c = h * w / g['dist']
                c = (c - 1.0) * p / (p + 1e-60) + 1.0
                u = u.clone()
                u[:, -1] = p / (GAMMA - 1) + ke + 1e-60
                new[ids] = u
                tau = taumin + c.abs() * tauscale
                sig = sigma0 / c.abs()
                gp = g['bcen'] + tau[:, None, None] * (cj - g['bcen'])
                avg = gp.mean(1, keepdim=True)
                span = torch.as_tensor(SPANS[g['t']], device=s0.device)
                pts = gp[:, span]
                det = torch.linalg.det(pts - avg[:, None])
                sub = (avg[:, None, 0] + pts.sum(2)) / (nd + 1)
                cnd = (sub * det[..., None]).sum(1) \
                    / det.sum(1, keepdim=True)
                idis = gp - cnd[:, None]
                jdis = gp - cj + (g['ccen'] - cnd)[:, None]
                udf = js + h * ut[j] - u[:, None] + torch.einsum(
                    'nfd,nfkd->nfk', jdis, j1)
                gr = torch.linalg.solve(idis[:, span], udf[:, span])
                wgt = 1.0 / torch.sqrt((gr * gr).sum(2) + 1e-200)
                ne = len(SPANS[g['t']])
                wgt = wgt / wgt.sum(1, keepdim=True) - 1.0 / ne
                hi = wgt.max(1).values.clamp(min=0.0)
                lo = wgt.min(1).values.clamp(max=0.0)
                sm = torch.minimum((1 - 1 / ne) / (hi + 1e-200),
                                   -1 / ne / (lo - 1e-200))
                sm = torch.minimum(sm, sig[:, None])
                wgt = 1.0 / ne + sm[:, None] * wgt
                grad[ids] = (wgt[:, :, None] * gr).sum(1).transpose(1, 2)
            g0 = self._ghost0(bc, pre)
            g1 = self._ghost1(bc, s1[:self.N])
            s0, s1 = torch.cat([new, g0]), torch.cat([grad, g1])
        return s0[:self.N], s1[:self.N]
