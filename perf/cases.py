"""Performance cases of the flux-reconstruction solver.

A case is one call that a flow simulation makes over and over: a time step
of an integrator (``run_steps``) or one evaluation of the semi-discrete
right-hand side (``system.rhs``), on the element types, orders, equations,
precisions and steppers the framework offers.  ``prepare`` makes what such a
program holds beforehand: the solver on its mesh (kept and given new initial
data, as a program that runs several initial conditions keeps it) with the
initial state on the GPU.  ``run`` is the call; its outputs are the solver's
own register banks, seen as tensors (in the banks' layout: blocks of 64
elements, and the elements of the last block that exist).

``exact`` evaluates the same discretisation in 64 bits from the mesh's
vertices and the published point sets alone: dense nodal operators from a
modal basis, faces paired by their flux points' coordinates.
"""
import json
import math

import numpy as np
import torch

TWOPI = 2*math.pi
GAMMA, MU, PR = 1.4, 1/1600, 0.71
CPTW = 2.5                      # wall temperature: that of rho = 1, p = 1/1.4

# Shunn-Ham tetrahedron, Williams-Shunn triangle and prism and layered
# pyramid point sets by order: sizes of the tables that hold them
NUPTS = {'hex': lambda p: (p + 1)**3,
         'tet': lambda p: (p + 1)*(p + 2)*(p + 3)//6,
         'pri': lambda p: (p + 1)**2*(p + 2)//2,
         'pyr': lambda p: (p + 1)*(p + 2)*(2*p + 3)//6}
NFPTS = {'hex': lambda p: 6*(p + 1)**2,
         'tet': lambda p: 2*(p + 1)*(p + 2),
         'pri': lambda p: (p + 1)*(p + 2) + 3*(p + 1)**2,
         'pyr': lambda p: (p + 1)**2 + 2*(p + 1)*(p + 2)}
STAGES = {'rk4': 4, 'rk45': 5}


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def _case(name, mesh, n, order, system, precision, scheme, call='step',
          walls=False, skew=False):
    """mesh: hex, tet, pri, tetpri (the upper third of the box prisms) or
    pyr; n: cells per edge of the box.  walls: isothermal no-slip walls at
    both ends of y.  skew: straight-sided elements that are no
    parallelepipeds."""
    return {'name': name, 'mesh': mesh, 'n': n, 'order': order,
            'system': system, 'precision': precision, 'scheme': scheme,
            'call': call, 'walls': walls, 'skew': skew}


def listed():
    ns, eu = 'navier-stokes', 'euler'
    return [
        # the smallest runs: a coarse box, where launches count
        _case('euler-hex8-p2-f64-rk4', 'hex', 8, 2, eu, 'double', 'rk4'),
        # a convergence study's middle grid, an odd number of elements
        _case('ns-hex13-p3-f64-rk45', 'hex', 13, 3, ns, 'double', 'rk45'),
        # the headline: direct simulation of the Taylor-Green vortex
        _case('ns-hex48-p3-f64-rk45', 'hex', 48, 3, ns, 'double', 'rk45'),
        # the same in the precision form (FP32 right-hand side, FP64 state)
        _case('ns-hex48-p3-mixed-rk45', 'hex', 48, 3, ns, 'mixed', 'rk45'),
        # inviscid flow, low order on a fine grid
        _case('euler-hex48-p2-f64-rk4', 'hex', 48, 2, eu, 'double', 'rk4'),
        # high order in single precision, an odd grid
        _case('euler-hex27-p4-f32-rk4', 'hex', 27, 4, eu, 'single', 'rk4'),
        # a wall-bounded flow on skewed elements; what another time
        # integrator or a residual monitor calls
        _case('ns-hex12-p4-f64-walls-rhs', 'hex', 12, 4, ns, 'double',
              'rk45', call='rhs', walls=True, skew=True),
        # the unstructured benchmark: tetrahedra with a layer of prisms
        _case('euler-tetpri24-p4-f32-rk4', 'tetpri', 24, 4, eu, 'single',
              'rk4'),
        _case('euler-tet17-p3-f64-rhs', 'tet', 17, 3, eu, 'double', 'rk4',
              call='rhs'),
        _case('ns-tetpri11-p3-f64-rk45', 'tetpri', 11, 3, ns, 'double',
              'rk45'),
        _case('euler-pyr18-p4-f32-rk4', 'pyr', 18, 4, eu, 'single', 'rk4'),
        # a low-order viscous run on tetrahedra in single precision
        _case('ns-tet9-p2-f32-walls-rk4', 'tet', 9, 2, ns, 'single', 'rk4',
              walls=True),
    ]


# cells per edge (the largest holds about 35 M unknowns on hexes) by order
_NMAX = {'hex': {1: 64, 2: 56, 3: 48, 4: 36},
         'tet': {1: 24, 2: 24, 3: 22, 4: 22},
         'tetpri': {1: 24, 2: 24, 3: 22, 4: 22},
         'pri': {1: 32, 2: 28, 3: 24, 4: 20},
         'pyr': {1: 22, 2: 20, 3: 18, 4: 17}}


def draw(rng):
    mesh = rng.choice(['hex', 'hex', 'hex', 'tet', 'tetpri', 'pri', 'pyr'])
    order = rng.randint(1, 4)
    system = rng.choice(['euler', 'navier-stokes'])
    precision = rng.choice(['double', 'double', 'single', 'mixed'])
    if mesh != 'hex' and precision == 'mixed':
        precision = 'single'
    call = rng.choice(['step', 'step', 'step', 'rhs'])
    if precision == 'mixed':
        call = 'step'
    walls = precision != 'mixed' and system == 'navier-stokes' and \
        rng.random() < 0.3
    skew = mesh == 'hex' and order > 1 and precision != 'mixed' and \
        rng.random() < 0.25
    hi = 12 if skew else _NMAX[mesh][order]
    n = round(math.exp(rng.uniform(math.log(4), math.log(hi))))
    c = _case('', mesh, n, order, system, precision,
              rng.choice(['rk4', 'rk45']), call, walls, skew)
    del c['name']
    return c


# ---------------------------------------------------------------------------
# The solver and its state
# ---------------------------------------------------------------------------

def _skew(x, y, z):
    """A smooth map of the box onto itself that keeps its sides."""
    s = 0.08*np.sin(x)*np.sin(y)*np.sin(z)
    return x + s, y - 0.7*s, z + 0.5*s


def _mesh(case):
    from pyfr_amd.mesh import BoxMesh, SimplexBoxMesh
    n = case['n']
    per = (True, not case['walls'], True)
    if case['mesh'] == 'hex':
        return BoxMesh(n, periodic=per, warp=_skew if case['skew'] else None)
    if case['mesh'] == 'tetpri':
        m = max(1, n//3)
        layers = [('tet', n - m), ('pri', m)]
    else:
        layers = [(case['mesh'], n)]
    return SimplexBoxMesh([((n, n, n), TWOPI/n, layers)], periodic=per)


def _dt(case):
    """A stable step (sound speed 1, flow speeds below 0.4)."""
    h = TWOPI/case['n']*(1.0 if case['mesh'] in ('hex', 'pri') else 0.3)
    dt = 0.15*h/((case['order'] + 1)**2)
    if case['system'] == 'navier-stokes':
        dt = min(dt, 0.02*(h/(case['order'] + 1)**2)**2/MU)
    return dt


def _cfg(case):
    from pyfr_amd.cases import make_cfg
    cfg = make_cfg(case['system'], case['order'], 'rusanov',
                   precision=case['precision'], scheme=case['scheme'],
                   dt=_dt(case))
    for k, v in (('rho', '1'), ('u', '0'), ('v', '0'), ('w', '0'),
                 ('p', repr(1/GAMMA))):
        cfg.set('soln-ics', k, v)
    if case['walls']:
        for side in ('y0', 'y1'):
            cfg.set(f'soln-bcs-{side}', 'type', 'no-slp-isot-wall')
            cfg.set(f'soln-bcs-{side}', 'cpTw', repr(CPTW))
    return cfg


class _Memory:
    """A typed window onto device memory of the solver."""

    def __init__(self, ptr, count, dtype):
        self.__cuda_array_interface__ = {
            'shape': (count,), 'typestr': np.dtype(dtype).str,
            'data': (int(ptr), False), 'version': 2}


def _views(mat):
    """The bank's values as tensors on its own memory: (points, variables,
    whole blocks, 64), and (points, variables, elements of the last block)
    where that block is not full."""
    nupts, nvar, neles = mat.ioshape
    flat = torch.as_tensor(_Memory(mat.data, mat.nrow*mat.leaddim,
                                   mat.dtype), device='cuda')
    nb, rem = divmod(neles, 64)
    out = []
    if nb:
        out.append(flat.as_strided((nupts, nvar, nb, 64),
                                   (mat.leaddim, 64, 64*nvar, 1)))
    if rem:
        out.append(flat.as_strided((nupts, nvar, rem),
                                   (mat.leaddim, 64, 1), nb*64*nvar))
    return out


class _Solver:
    """A solver on a case's mesh, kept between initial states."""

    def __init__(self, case):
        from pyfr_amd.backend import AMDBackend
        from pyfr_amd.solvers import get_integrator
        cfg = _cfg(case)
        self.backend = AMDBackend(cfg)
        self.integ = get_integrator(self.backend, _mesh(case), cfg)
        system = self.integ.system
        self.coords = [torch.as_tensor(np.ascontiguousarray(
            e.geom.ploc_at(e.basis.upts)), device='cuda')
            for e in system.ele_map.values()]
        self.views = [[_views(b) for b in banks]
                      for banks in system.ele_banks]

    def set_state(self, case, seed):
        integ = self.integ
        arrs = [_initial(case, seed, x).cpu().numpy() for x in self.coords]
        integ.system.set_soln_upts(integ.idxcurr, arrs)
        if case['precision'] == 'mixed':
            integ._work_valid = False   # the FP32 copy of the old state


class _State:
    """A solver with one initial state; gives the solver back when it goes."""

    def __init__(self, key, solver, case):
        self.key, self.solver, self.call = key, solver, case['call']

    def __del__(self):
        if _idle and self.key in _idle:
            _idle[self.key].append(self.solver)


_idle = {}                      # solvers of the present case that are free


def prepare(case, seed):
    case = {k: v for k, v in case.items() if k != 'name'}
    key = json.dumps(case, sort_keys=True)
    if key not in _idle:
        _idle.clear()
        _idle[key] = []
    solver = _idle[key].pop() if _idle[key] else _Solver(case)
    solver.set_state(case, seed)
    return _State(key, solver, case)


def run(state):
    integ = state.solver.integ
    if state.call == 'rhs':
        out = 1 - integ.idxcurr
        integ.system.rhs(integ.tcurr, integ.idxcurr, out)
    else:
        integ.run_steps(1)
        out = integ.idxcurr
    return [v[out] for v in state.solver.views]


def _initial(case, seed, x):
    """Conserved variables (points, 5, elements) at coordinates x (points,
    3, elements): a Taylor-Green vortex and four random modes, their sum
    brought to rest at walls."""
    rng = np.random.default_rng(seed)
    X = x[:, 0], x[:, 1], x[:, 2]
    a, b, c = (x[:, i] + s for i, s in enumerate(rng.uniform(0, TWOPI, 3)))
    amp = 0.1*rng.uniform(0.8, 1.2)
    vel = [amp*torch.sin(a)*torch.cos(b)*torch.cos(c),
           -amp*torch.cos(a)*torch.sin(b)*torch.cos(c),
           torch.zeros_like(a)]
    rho = torch.ones_like(a)
    p = 1/GAMMA + amp*amp*(torch.cos(2*a) + torch.cos(2*b)) * \
        (torch.cos(2*c) + 2)/16
    for _ in range(4):
        k = rng.integers(1, 3, 3)*rng.choice([-1, 1], 3)
        w = torch.sin(sum(int(ki)*xi for ki, xi in zip(k, X)) +
                      rng.uniform(0, TWOPI))
        rho = rho + 0.02*w*rng.uniform(0.5, 1)
        for i, v in enumerate(rng.uniform(-0.02, 0.02, 3)):
            vel[i] = vel[i] + v*w
    if case['walls']:
        vel = [v*torch.sin(X[1]/2) for v in vel]
    E = p/(GAMMA - 1) + 0.5*rho*(vel[0]**2 + vel[1]**2 + vel[2]**2)
    return torch.stack([rho, *(rho*v for v in vel), E], dim=1)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far results may differ
# ---------------------------------------------------------------------------

def _blocks(case):
    """(element type, elements) of the mesh."""
    n = case['n']
    if case['mesh'] == 'tetpri':
        m = max(1, n//3)
        return [('tet', 6*n*n*(n - m)), ('pri', 2*n*n*m)]
    per = {'hex': 1, 'tet': 6, 'pri': 2, 'pyr': 6}[case['mesh']]
    return [(case['mesh'], per*n**3)]


def work(case):
    """Each evaluation of the right-hand side reads the state and writes its
    result (or, in a step, the next stage's state), and interface values
    cross from element to element once: one value of each variable at each
    flux point written and read (twice for Navier-Stokes: the gradients need
    the common solution first).  Operations are those of the dense (for hexes:
    line by line) operators and some 150 a point for the fluxes."""
    p, ns = case['order'], case['system'] == 'navier-stokes'
    isz = 8 if case['precision'] == 'double' else 4
    nb = nf = 0.0
    for et, ne in _blocks(case):
        nu, nfp = NUPTS[et](p), NFPTS[et](p)
        nb += ne*5*isz*(2*nu + 2*nfp*(2 if ns else 1))
        if et == 'hex':
            mm = 3*nu*(p + 1) + 2*3*nu + nfp*(p + 1)
        else:
            mm = nu*(3*nu + nfp) + nfp*nu
        nf += ne*(2*5*mm*(2.6 if ns else 1) + 150*(nu + nfp)*(2 if ns else 1))
    stages = 1 if case['call'] == 'rhs' else STAGES[case['scheme']]
    return {'bytes': nb*stages, 'flops': nf*stages}


def tolerance(case):
    """Right-hand sides are sums of fluxes that cancel: they keep fewer
    digits than the state they are computed from."""
    if case['call'] == 'rhs':
        return ({'rel': 2e-10, 'max': 5e-9} if case['precision'] == 'double'
                else {'rel': 1e-3, 'max': 1e-2})
    return {'double': {'rel': 2e-13, 'max': 5e-12},
            'mixed': {'rel': 2e-6, 'max': 5e-5},
            'single': {'rel': 5e-7, 'max': 3e-6}}[case['precision']]


# ---------------------------------------------------------------------------
# The same discretisation in 64 bits
# ---------------------------------------------------------------------------

def _gl(n):
    return np.polynomial.legendre.leggauss(n)


def _leg(kmax, x):
    """Legendre polynomials and derivatives: two (kmax + 1, npts) arrays."""
    P, D = [np.ones_like(x), x], [np.zeros_like(x), np.ones_like(x)]
    for k in range(2, kmax + 1):
        P.append(((2*k - 1)*x*P[-1] - (k - 1)*P[-2])/k)
        D.append((2*k - 1)*P[k - 1] + D[k - 2])
    return P, D


def _cone(kmax, x, s):
    """s^k P_k(x/s) and its derivatives along x and s."""
    one, nil = np.ones_like(x), np.zeros_like(x)
    Q, X, S = [one, x], [nil, one], [nil, nil]
    for k in range(2, kmax + 1):
        a, b = (2*k - 1)/k, (k - 1)/k
        Q.append(a*x*Q[k - 1] - b*s*s*Q[k - 2])
        X.append(a*(Q[k - 1] + x*X[k - 1]) - b*s*s*X[k - 2])
        S.append(a*x*S[k - 1] - b*(2*s*Q[k - 2] + s*s*S[k - 2]))
    return Q, X, S


def _basis(et, p, pts):
    """A basis of the element's space at pts: values (npts, nb) and
    derivatives (3, npts, nb)."""
    x, y, z = np.asarray(pts, dtype=float).T
    r = range(p + 1)
    if et == 'pyr':
        s = (1 - z)/2
        (A, Ax, As), (B, By, Bs) = _cone(p, x, s), _cone(p, y, s)
        C, Cz = _leg(p, z)
        t = [(i, j, k) for i in r for j in r for k in range(p + 1 - max(i, j))]
        val = [A[i]*B[j]*C[k] for i, j, k in t]
        dx = [Ax[i]*B[j]*C[k] for i, j, k in t]
        dy = [A[i]*By[j]*C[k] for i, j, k in t]
        dz = [-0.5*(As[i]*B[j] + A[i]*Bs[j])*C[k] + A[i]*B[j]*Cz[k]
              for i, j, k in t]
    else:
        keep = {'hex': lambda i, j, k: True, 'tet': lambda i, j, k:
                i + j + k <= p, 'pri': lambda i, j, k: i + j <= p}[et]
        t = [(i, j, k) for i in r for j in r for k in r if keep(i, j, k)]
        (A, Ax), (B, By), (C, Cz) = (_leg(p, v) for v in (x, y, z))
        val = [A[i]*B[j]*C[k] for i, j, k in t]
        dx = [Ax[i]*B[j]*C[k] for i, j, k in t]
        dy = [A[i]*By[j]*C[k] for i, j, k in t]
        dz = [A[i]*B[j]*Cz[k] for i, j, k in t]
    return np.array(val).T, np.array([dx, dy, dz]).transpose(0, 2, 1)


def _quadrature(et, n):
    """Points and weights, exact for the products of basis functions."""
    g, w = _gl(n)
    a, b, c = (v.ravel() for v in np.meshgrid(g, g, g, indexing='ij'))
    wt = np.einsum('i,j,k->ijk', w, w, w).ravel()
    if et == 'pyr':
        s = (1 - c)/2
        return np.stack([s*a, s*b, c], 1), wt*s*s
    if et in ('tet', 'pri'):        # collapse x onto y, then both onto z
        a, wt = (1 + a)*(1 - b)/2 - 1, wt*(1 - b)/2
    if et == 'tet':
        s = (1 - c)/2
        return np.stack([(1 + a)*s - 1, (1 + b)*s - 1, c], 1), wt*s*s
    return np.stack([a, b, c], 1), wt


def _face_basis(kind, p, st):
    (A, _), (B, _) = (_leg(p, v) for v in np.asarray(st, dtype=float).T)
    return np.array([A[i]*B[j] for i in range(p + 1) for j in range(p + 1)
                     if kind == 'quad' or i + j <= p]).T


VERTS = {'hex': [(x, y, z) for z in (-1, 1) for y in (-1, 1) for x in (-1, 1)],
         'tet': [(-1, -1, -1), (1, -1, -1), (-1, 1, -1), (-1, -1, 1)],
         'pri': [(x, y, z) for z in (-1, 1)
                 for x, y in ((-1, -1), (1, -1), (-1, 1))],
         'pyr': [(-1, -1, -1), (1, -1, -1), (-1, 1, -1), (1, 1, -1),
                 (0, 0, 1)]}
# corner, then its two neighbours on the face, of each face
FACES = {'hex': [(0, 1, 2), (4, 5, 6), (0, 1, 4), (2, 3, 6), (0, 2, 4),
                 (1, 3, 5)],
         'tet': [(0, 1, 2), (0, 1, 3), (0, 2, 3), (1, 2, 3)],
         'pri': [(0, 1, 2), (3, 4, 5), (0, 1, 3), (1, 2, 4), (0, 2, 3)],
         'pyr': [(0, 1, 2), (0, 1, 4), (1, 3, 4), (2, 3, 4), (0, 2, 4)]}
QUADS = {'hex': range(6), 'tet': (), 'pri': (2, 3, 4), 'pyr': (0,)}


def _upts(et, p):
    if et == 'hex':
        g = _gl(p + 1)[0]
        return np.array([(x, y, z) for z in g for y in g for x in g])
    from pyfr_amd.quadtables import TABLES      # the published point sets
    fam = {'tet': 'shunn-ham', 'pri': 'williams-shunn~gauss-legendre',
           'pyr': 'gauss-legendre'}[et]
    return np.array(TABLES[et, fam, NUPTS[et](p)][0])


class _Element:
    """Operators of one element type, on the GPU in 64 bits."""

    def __init__(self, et, p, verts):
        from pyfr_amd.quadtables import TABLES
        upts = _upts(et, p)
        V, dV = _basis(et, p, upts)
        Vi = np.linalg.inv(V)
        qp, qw = _quadrature(et, 2*p + 4)
        B = _basis(et, p, qp)[0]
        proj = V @ np.linalg.inv((B*qw[:, None]).T @ B)
        rv = np.array(VERTS[et], dtype=float)
        fpts, norms, lift = [], [], []
        for f, (a, b, c) in enumerate(FACES[et]):
            kind = 'quad' if f in QUADS[et] else 'tri'
            va, ds, dt = rv[a], (rv[b] - rv[a])/2, (rv[c] - rv[a])/2
            n = np.cross(ds, dt)
            if n @ (va + ds + dt - rv.mean(axis=0)) < 0:
                n = -n
            g, w = _gl(2*p + 4)
            s, t = (v.ravel() for v in np.meshgrid(g, g, indexing='ij'))
            w = np.outer(w, w).ravel()
            if kind == 'tri':
                s, w = (1 + s)*(1 - t)/2 - 1, w*(1 - t)/2
                st = np.array(TABLES['tri', 'williams-shunn',
                                     (p + 1)*(p + 2)//2][0])
            else:
                st = np.array([(x, y) for y in _gl(p + 1)[0]
                               for x in _gl(p + 1)[0]])
            at = lambda q: va + (q[:, :1] + 1)*ds + (q[:, 1:] + 1)*dt
            q = np.stack([s, t], 1)
            L = _face_basis(kind, p, q) @ np.linalg.inv(
                _face_basis(kind, p, st))
            lift.append(proj @ (_basis(et, p, at(q))[0]*w[:, None]).T @ L)
            fpts.append(at(st))
            norms.append(np.tile(n, (len(st), 1)))
        fpts = np.concatenate(fpts)
        dev = lambda m: torch.as_tensor(np.ascontiguousarray(m),
                                        device='cuda')
        self.to_f = dev(_basis(et, p, fpts)[0] @ Vi)
        self.diff = [dev(d @ Vi) for d in dV]
        self.lift = dev(np.concatenate(lift, axis=1))
        self.norm = dev(np.concatenate(norms))
        self.nu, self.nf, self.ne = len(upts), len(fpts), verts.shape[1]
        v = dev(verts)                                  # (nverts, ne, 3)
        self.x, S, J = self._metric(et, v, upts)
        self.xf, Sf, _ = self._metric(et, v, fpts)
        self.S, self.J = S, J
        # unnormalised physical normals (3, nf, ne)
        self.nrm = sum(self.norm[:, i, None]*Sf[i] for i in range(3))

    @staticmethod
    def _metric(et, v, pts):
        """Coordinates (npts, 3, ne); S[i][k] = |J| dxi_i/dx_k; |J|."""
        q = torch.as_tensor(np.asarray(pts, dtype=float), device='cuda')
        if et == 'hex':
            sg = torch.as_tensor(np.array(VERTS['hex'], dtype=float),
                                 device='cuda')
            f = 1 + q[:, None, :]*sg[None]              # (npts, 8, 3)
            N = f.prod(dim=2)/8
            dN = [sg[:, 0]*f[:, :, 1]*f[:, :, 2]/8,
                  sg[:, 1]*f[:, :, 0]*f[:, :, 2]/8,
                  sg[:, 2]*f[:, :, 0]*f[:, :, 1]/8]
            x = torch.stack([N @ v[:, :, b] for b in range(3)], 1)
            j = [[d @ v[:, :, b] for b in range(3)] for d in dN]
        else:
            # the affine map of the corners next to the first
            e = [(v[1] - v[0])/2, (v[2] - v[0])/2,
                 (v[4] - (v[1] + v[2])/2)/2 if et == 'pyr'
                 else (v[3] - v[0])/2]
            ones = torch.ones_like(q[:, :1])
            j = [[ones*e[a][:, b] for b in range(3)] for a in range(3)]
            x = torch.stack([v[0][:, b] + sum((q[:, a:a + 1] + 1) *
                             e[a][:, b] for a in range(3))
                             for b in range(3)], 1)
        S = []
        for a, b in ((1, 2), (2, 0), (0, 1)):
            S.append(torch.stack([
                j[a][1]*j[b][2] - j[a][2]*j[b][1],
                j[a][2]*j[b][0] - j[a][0]*j[b][2],
                j[a][0]*j[b][1] - j[a][1]*j[b][0]]))
        return x, S, sum(j[0][k]*S[0][k] for k in range(3))

    def op(self, m, u):
        return (m @ u.reshape(u.shape[0], -1)).reshape(m.shape[0],
                                                       *u.shape[1:])


def _inviscid(u):
    """Flux f[k] (5, ...) of the state u[0..4], pressure and velocity."""
    v = [u[i]/u[0] for i in (1, 2, 3)]
    p = (GAMMA - 1)*(u[4] - 0.5*(u[1]*v[0] + u[2]*v[1] + u[3]*v[2]))
    f = []
    for k in range(3):
        c = [u[k + 1], *(u[i + 1]*v[k] for i in range(3)), (u[4] + p)*v[k]]
        c[k + 1] = c[k + 1] + p
        f.append(c)
    return f, p, v


def _viscous(u, g):
    """Viscous flux f[k] (5, ...) from physical gradients g[k][var]."""
    v = [u[i]/u[0] for i in (1, 2, 3)]
    dv = [[(g[k][i + 1] - v[i]*g[k][0])/u[0] for k in range(3)]
          for i in range(3)]                            # dv_i/dx_k
    div = dv[0][0] + dv[1][1] + dv[2][2]
    f = []
    for k in range(3):
        tau = [MU*(dv[i][k] + dv[k][i] - (2/3*div if i == k else 0))
               for i in range(3)]
        de = (g[k][4] - u[4]/u[0]*g[k][0])/u[0] - \
            sum(v[i]*dv[i][k] for i in range(3))
        f.append([0*de, *(-t for t in tau), -MU*GAMMA/PR*de -
                  sum(v[i]*tau[i] for i in range(3))])
    return f


def _rusanov(ul, ur, n):
    (fl, pl, vl), (fr, pr, vr) = _inviscid(ul), _inviscid(ur)
    nv = sum(n[k]*(vl[k] + vr[k]) for k in range(3))
    a = torch.sqrt(0.25*GAMMA*(pl + pr)/(ul[0] + ur[0])) + 0.25*nv.abs()
    return [0.5*sum(n[k]*(fl[k][i] + fr[k][i]) for k in range(3)) +
            a*(ul[i] - ur[i]) for i in range(5)]


class _Exact:
    def __init__(self, case):
        mesh = _mesh(case)
        self.ns = case['system'] == 'navier-stokes'
        self.walls = case['walls']
        self.eles = [_Element(et, case['order'], v)
                     for et, v in mesh.spts.items()]
        xf = torch.cat([e.xf.transpose(1, 2).reshape(-1, 3)
                        for e in self.eles])
        self.nrm = torch.cat([e.nrm.reshape(3, -1) for e in self.eles], 1)
        self.mag = torch.sqrt((self.nrm**2).sum(dim=0))
        self.unit = self.nrm/self.mag
        wall = torch.zeros(len(xf), dtype=torch.bool, device='cuda')
        if self.walls:
            wall = (xf[:, 1].abs() < 1e-9) | ((xf[:, 1] - TWOPI).abs() < 1e-9)
        # points of one place share a key; periodic images fold together
        other = torch.arange(len(xf), device='cuda')
        todo = other[~wall]
        for off in (0.0123, 0.00317):
            q = torch.round(torch.remainder(xf[todo] + off, TWOPI)/1e-5)
            q = torch.remainder(q.long(), round(TWOPI/1e-5))
            key = (q[:, 0]*700001 + q[:, 1])*700001 + q[:, 2]
            key, order = torch.sort(key)
            same = (key[1:] == key[:-1]).nonzero()[:, 0]
            a, b = todo[order[same]], todo[order[same + 1]]
            other[a], other[b] = b, a
            todo = todo[other[todo] == todo]
        if len(todo):
            raise RuntimeError('faces do not pair')
        self.other, self.wall = other, wall

    def _join(self, fs):
        """Per-element arrays (nf, nvar, ne) as a list of nvar flat ones."""
        return [torch.cat([f[:, v].reshape(-1) for f in fs])
                for v in range(fs[0].shape[1])]

    def _split(self, flat):
        out, at = [], 0
        for e in self.eles:
            m = e.nf*e.ne
            out.append(torch.stack([f[at:at + m].reshape(e.nf, e.ne)
                                    for f in flat], 1))
            at += m
        return out

    def rhs(self, us):
        uf = [e.op(e.to_f, u) for e, u in zip(self.eles, us)]
        ul = self._join(uf)
        ur = [x[self.other] for x in ul]
        uw = None
        if self.walls:
            w = self.wall
            zero = torch.zeros_like(ul[0])
            uw = [ul[0], zero, zero, zero, CPTW/GAMMA*ul[0]]
            ke = 0.5*(ul[1]**2 + ul[2]**2 + ul[3]**2)/ul[0]
            gh = [ul[0], -ul[1], -ul[2], -ul[3], CPTW/GAMMA*ul[0] + ke]
            ur = [torch.where(w, a, b) for a, b in zip(gh, ur)]
        fn = _rusanov(ul, ur, self.unit)
        grads = [None]*len(us)
        if self.ns:
            com = [0.5*(a + b) for a, b in zip(ul, ur)]
            if self.walls:
                com = [torch.where(self.wall, a, b) for a, b in zip(uw, com)]
            gf = []
            for i, (e, u, c, f) in enumerate(zip(self.eles, us,
                                                 self._split(com), uf)):
                gr = [e.op(e.diff[d], u) +
                      e.op(e.lift, e.norm[:, d, None, None]*(c - f))
                      for d in range(3)]
                g = [sum(e.S[d][k][:, None]*gr[d] for d in range(3)) /
                     e.J[:, None] for k in range(3)]
                grads[i] = g
                gf.append([e.op(e.to_f, x) for x in g])
            gl = [self._join([g[k] for g in gf]) for k in range(3)]
            ub = ul if uw is None else [torch.where(self.wall, a, b)
                                        for a, b in zip(uw, ul)]
            fv = _viscous(ub, gl)
            nl = [sum(self.unit[k]*fv[k][i] for k in range(3))
                  for i in range(5)]
            # seen from the other side the normal points the other way
            both = [0.5*(x - x[self.other]) for x in nl]
            if self.walls:
                both = [torch.where(self.wall, a, b)
                        for a, b in zip(nl, both)]
            fn = [a + b for a, b in zip(fn, both)]
        fn = self._split([self.mag*x for x in fn])
        out = []
        for e, u, c, g in zip(self.eles, us, fn, grads):
            f, _, _ = _inviscid(u.unbind(1))
            if g is not None:
                fv = _viscous(u.unbind(1), [x.unbind(1) for x in g])
                f = [[a + b for a, b in zip(x, y)] for x, y in zip(f, fv)]
            f = [torch.stack(x, 1) for x in f]
            F = [sum(e.S[d][k][:, None]*f[k] for k in range(3))
                 for d in range(3)]
            r = sum(e.op(e.diff[d], F[d]) for d in range(3))
            own = sum(e.norm[:, d, None, None]*e.op(e.to_f, F[d])
                      for d in range(3))
            r = r + e.op(e.lift, c - own)
            out.append(-r/e.J[:, None])
        return out


# Kennedy, Carpenter and Lewis' low-storage five-stage scheme (2R+)
RK45_A = [970286171893 / 4311952581923, 6584761158862 / 12103376702013,
          2251764453980 / 15575788980749, 26877169314380 / 34165994151039]
RK45_B = [1153189308089 / 22510343858157, 1772645290293 / 4653164025191,
          -1672844663538 / 4480602732383, 2114624349019 / 3568978502595,
          5198255086312 / 14908931495163]


def _axpy(a, xs, ys):
    return [y + a*x for x, y in zip(xs, ys)]


def exact(case, seed):
    ex = _Exact(case)
    us = [_initial(case, seed, e.x) for e in ex.eles]
    if case['precision'] == 'single':
        us = [u.float().double() for u in us]
    dt = _dt(case)
    if case['call'] == 'rhs':
        us = ex.rhs(us)
    elif case['scheme'] == 'rk4':
        k1 = ex.rhs(us)
        k2 = ex.rhs(_axpy(dt/2, k1, us))
        k3 = ex.rhs(_axpy(dt/2, k2, us))
        k4 = ex.rhs(_axpy(dt, k3, us))
        for a, k in ((dt/6, k1), (dt/3, k2), (dt/3, k3), (dt/6, k4)):
            us = _axpy(a, k, us)
    else:
        acc, cur = us, us
        for i, b in enumerate(RK45_B):
            k = ex.rhs(cur)
            if i < 4:
                cur = _axpy(dt*RK45_A[i], k, acc)
            acc = _axpy(dt*b, k, acc)
        us = acc
    if case['precision'] == 'mixed':
        # its register holds the state less the constant state at rest
        rest = torch.zeros(5, dtype=torch.float64, device='cuda')
        rest[0], rest[4] = 1.0, 1/GAMMA/(GAMMA - 1)
        us = [u - rest[:, None] for u in us]
    out = []
    for u in us:
        nb, rem = divmod(u.shape[2], 64)
        parts = []
        if nb:
            parts.append(u[:, :, :64*nb].reshape(u.shape[0], 5, nb, 64))
        if rem:
            parts.append(u[:, :, 64*nb:])
        out.append(parts)
    return out
