"""Line kernels of hexahedra: their 1-D operators against the full ones, and
the passes that run in them against the kernel sequences they replace."""
import numpy as np
import pytest

from pyfr_amd.mesh import BoxMesh
from pyfr_amd.shapes import HEX_FACES, HexShape
from pyfr_amd.solvers import get_integrator
from tests.fr_cases import make_cfg, rel_l2


@pytest.mark.parametrize('order', [1, 2, 3, 4])
def test_lines_make_the_operators(order):
    """M0, M3, M6 and the corrected derivatives, rebuilt from the lines."""
    sh = HexShape(order)
    d, hl, hr, ll, lr, _ = sh.lines
    n, nu = sh.n, sh.nupts
    m0, m3 = np.zeros((sh.nfpts, nu)), np.zeros((nu, sh.nfpts))
    m6 = np.zeros((3*nu, sh.nfpts))
    for f, (nax, side, _, _) in enumerate(HEX_FACES):
        for b in range(n):
            for a in range(n):
                line, row = sh.fpt_line(f, a, b)[0], f*n*n + a + n*b
                m0[row, line] = lr if side > 0 else ll
                m3[line, row] = hr if side > 0 else hl
                m6[nax*nu + np.array(line), row] = side*m3[line, row]
    div = np.zeros((nu, 3*nu))
    for p in range(nu):
        c = [p % n, p//n % n, p//(n*n)]
        for ax in range(3):
            for m in range(n):
                q = list(c)
                q[ax] = m
                div[p, ax*nu + sh.uidx(*q)] = d[c[ax], m]
    grad = div.reshape(nu, 3, nu).swapaxes(0, 1).reshape(3*nu, nu)
    for got, expr in ((m0, 'M0'), (m3, 'M3'), (m6, 'M6'),
                      (div, 'M1 - M3*M2'), (grad, 'M4 - M6*M0')):
        ref = sh.opmat(expr)
        # sums of a few products of entries up to about 30
        assert np.abs(got - ref).max() < 1e-13, expr


def _warp(x, y, z):
    """Moves the low-x half only: curved elements there, linear beyond."""
    s = np.where(x < 3.0, 0.05*np.sin(x)**2*np.sin(y)*np.sin(z), 0.0)
    return x + s, y - s, z + 0.5*s


def _run(make, system, n, order, fuse, scheme=None, steps=2, kind='straight',
         precision='double', **cfgkw):
    be = make(precision=precision, fuse_flux=fuse)
    consts = cfgkw.pop('constants', {})
    cfg = make_cfg(system, order, precision=precision,
                   scheme=scheme or 'rk4', dt=1e-3, **cfgkw)
    for k, v in consts.items():
        cfg.set('constants', k, v)
    kw = {}
    if kind == 'skew':
        kw = {'warp': lambda x, y, z: (x + 0.05*np.sin(y), y, z)}
    elif kind == 'mixed':
        kw = {'sorder': 2, 'warp': _warp}
    integ = get_integrator(be, BoxMesh(n, **kw), cfg)
    sysm = integ.system
    if scheme is None:
        sysm.rhs(0.0, 0, 1)
        return sysm.ele_scal_upts(1)[0], sysm
    integ.run_steps(steps, 1e-3)
    return integ.soln[0], sysm


def _rms(a):
    return float(np.sqrt(np.mean(np.square(a))))


def _rounding(n, order):
    """Rounding error of a right-hand side: its terms are fluxes of up to
    250 (of E, at p = 71.5) times 2/h = n/pi times 1-D derivatives whose
    rows sum to 2(p + 1)^2 in modulus; eight roundings of each."""
    return 8*2.2e-16*250*max(n)/np.pi*2*(order + 1)**2


# 60 elements end in a partial block; the larger meshes reach the blocks of
# more than 16 elements that grids of 256 blocks and over take
SIZES = [((5, 4, 3), o) for o in (1, 2, 3, 4)] + \
        [((26, 26, 25), 1), ((26, 26, 25), 2)]


@pytest.mark.gpu
@pytest.mark.parametrize('n,order,kind', [
    (n, o, k) for n, o in SIZES for k in ('straight', 'skew')] + [
    ((6, 6, 6), 2, 'mixed'), ((6, 6, 6), 3, 'mixed')])
def test_euler_rhs(backend_factory, n, order, kind):
    """Flux, divergence and correction in one kernel, on straight, skewed
    and part curved meshes."""
    print(f'\n[hexline rhs] {n} p={order} {kind}', flush=True)
    got, sysm = _run(backend_factory, 'euler', n, order, True, kind=kind)
    ref, _ = _run(backend_factory, 'euler', n, order, False, kind=kind)
    if kind == 'mixed':
        assert len(sysm.ele_map['hex'].mesh_regions) == 2
    assert _rms(got - ref) < _rounding(n, order)


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['rk4', 'rk45', 'rk34', 'euler'])
@pytest.mark.parametrize('precision', ['double', 'single', 'mixed'])
@pytest.mark.parametrize('n,order', [((5, 4, 3), 1), ((5, 4, 3), 3),
                                     ((21, 21, 19), 4), ((26, 26, 25), 3)])
def test_euler_steps(backend_factory, scheme, precision, n, order):
    """The stage updates, and the traces of the next stage's input left by
    the kernel that forms it."""
    if precision == 'mixed' and scheme == 'euler':
        pytest.skip('no such stepper')
    if n[0] > 5 and (precision == 'double' or scheme in ('rk34', 'euler')):
        pytest.skip('these blocks are only taken in single precision')
    print(f'\n[hexline step] {n} p={order} {scheme} {precision}', flush=True)
    got, _ = _run(backend_factory, 'euler', n, order, True, scheme,
                  precision=precision)
    ref, _ = _run(backend_factory, 'euler', n, order, False, scheme,
                  precision=precision)
    # two steps: rounding of the state, and the right-hand side's in dt
    tol = {'double': 1e-14, 'single': 2e-6, 'mixed': 1e-6}[precision]
    assert rel_l2(got, ref) < tol


@pytest.mark.gpu
@pytest.mark.parametrize('n,order,kind', [
    ((5, 4, 3), o, k) for o in (1, 2, 3, 4) for k in ('straight', 'skew')] + [
    ((6, 6, 6), 2, 'mixed'), ((6, 6, 6), 3, 'mixed')])
@pytest.mark.parametrize('beta,tau,visc', [(0.0, 0.0, 'none'),
                                           (0.5, 0.1, 'none'),
                                           (-0.5, 0.0, 'none'),
                                           (0.25, 0.1, 'none')])
def test_ns_rhs(backend_factory, n, order, kind, beta, tau, visc):
    """Gradient, flux and divergence in one kernel; linear meshes pass the
    interfaces each side's normal viscous flux, part curved ones (and p = 1,
    whose metric is stored) the gradients."""
    print(f'\n[hexline ns] {n} p={order} {kind} {beta} {tau}', flush=True)
    kw = dict(kind=kind, beta=beta, tau=tau, visc_corr=visc)
    got, sysm = _run(backend_factory, 'navier-stokes', n, order, True, **kw)
    assert sysm._nfv == (kind != 'mixed' and order > 1)
    ref, _ = _run(backend_factory, 'navier-stokes', n, order, False, **kw)
    # the viscous terms, a second derivative of fluxes of mu times order 1,
    # stay below the inviscid ones
    assert _rms(got - ref) < _rounding(n, order)


# c_p T of the field is about 250
SUTHERLAND = {'mu': 0.02, 'cpTref': 250.0, 'cpTs': 110.0}


@pytest.mark.gpu
@pytest.mark.parametrize('n,order,kind', [
    ((5, 4, 3), o, k) for o in (1, 2, 3, 4) for k in ('straight', 'skew')] + [
    ((6, 6, 6), 2, 'mixed'), ((6, 6, 6), 3, 'mixed')])
@pytest.mark.parametrize('beta,tau', [(0.0, 0.0), (0.25, 0.1)])
def test_ns_sutherland(backend_factory, n, order, kind, beta, tau):
    """Temperature-dependent viscosity, inside the elements and in the
    normal viscous flux (straight, skew) or the gradients (mixed, p = 1)
    that the interfaces get."""
    print(f'\n[hexline sutherland] {n} p={order} {kind} {beta}', flush=True)
    kw = dict(kind=kind, beta=beta, tau=tau, constants=SUTHERLAND)
    got, sysm = _run(backend_factory, 'navier-stokes', n, order, True,
                     visc_corr='sutherland', **kw)
    assert sysm._nfv == (kind != 'mixed' and order > 1)
    ref, _ = _run(backend_factory, 'navier-stokes', n, order, False,
                  visc_corr='sutherland', **kw)
    assert _rms(got - ref) < _rounding(n, order)
    plain, _ = _run(backend_factory, 'navier-stokes', n, order, True,
                    visc_corr='none', **kw)
    assert _rms(got - plain) > 1e6*_rounding(n, order)


@pytest.mark.gpu
@pytest.mark.parametrize('fuse', [True, False])
@pytest.mark.parametrize('order', [1, 2, 3])
def test_sutherland_oracle(backend_factory, fuse, order):
    """The same against the oracle, in the one-pass kernels and in those
    they replace."""
    from oracle.rhs import OracleHexSystem
    from tests.fr_cases import oracle_consts
    from tests.test_gpu_parity import rhs_noise_floor
    print(f'\n[hexline sutherland oracle] p={order} {fuse}', flush=True)
    got, _ = _run(backend_factory, 'navier-stokes', 3, order, fuse,
                  visc_corr='sutherland', constants=SUTHERLAND)
    orc = OracleHexSystem(3, order, 'navier-stokes', constants=oracle_consts(
        'navier-stokes') | SUTHERLAND | {'visc_corr': 'sutherland'})
    u0 = orc.ics()
    err = rel_l2(got, orc.rhs(u0))
    tol = max(1e-12, 10*rhs_noise_floor(orc, u0))
    print(f'[hexline sutherland oracle] rel L2 {err:.3e} (tol {tol:.3e})',
          flush=True)
    assert err < tol


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['rk4', 'rk45'])
@pytest.mark.parametrize('order', [1, 2])
def test_euler_steps_double_whole_blocks(backend_factory, scheme, order):
    """The stage updates and next-stage traces of the FP64 kernel with 64
    elements a block, which only grids of 256 blocks and over take."""
    n = (26, 26, 25)
    print(f'\n[hexline step 64] p={order} {scheme}', flush=True)
    got, _ = _run(backend_factory, 'euler', n, order, True, scheme)
    ref, _ = _run(backend_factory, 'euler', n, order, False, scheme)
    assert rel_l2(got, ref) < 1e-14


@pytest.mark.gpu
@pytest.mark.parametrize('scheme', ['rk4', 'rk45'])
@pytest.mark.parametrize('precision', ['double', 'single', 'mixed'])
@pytest.mark.parametrize('n,order', [((5, 4, 3), 2), ((5, 4, 3), 4),
                                     ((9, 8, 8), 3)])
def test_ns_steps(backend_factory, scheme, precision, n, order):
    print(f'\n[hexline ns step] {n} p={order} {scheme} {precision}',
          flush=True)
    got, _ = _run(backend_factory, 'navier-stokes', n, order, True, scheme,
                  precision=precision)
    ref, _ = _run(backend_factory, 'navier-stokes', n, order, False, scheme,
                  precision=precision)
    tol = {'double': 1e-14, 'single': 2e-6, 'mixed': 1e-6}[precision]
    assert rel_l2(got, ref) < tol


def _offset(x, y, z):
    return x + 100.0 + 0.05*np.sin(y), y - 100.0 + 0.03*np.sin(z), z + 50.0


@pytest.mark.parametrize('order', [2, 4])
def test_face_normals(monkeypatch, order):
    """The normals that the viscous flux at the interfaces is taken along:
    those of the stored metric, and in single precision one rounding of
    each coefficient from it, wherever the mesh lies."""
    import pyfr_amd._lib as _lib
    from pyfr_amd.backend import AMDBackend
    from tests.test_ns_options import StubLib
    monkeypatch.setattr(_lib, '_lib', StubLib())
    # 1.2e-7: half an ulp of each of three coefficients, the largest of them
    # the normal itself.  The stored metric's own rounding: it is a
    # derivative of X x X_a, which is a derivative too, in components of two
    # products of up to 106.3 and 1.05 (half an edge), on normals of 0.3 and
    # more; the derivative matrices' rows sum to at most 2 p^2 in modulus
    meps = 2.2e-16*2*106.3*1.05/0.3*(2*order*order)**2
    for precision, eps in (('double', meps), ('single', 1.2e-7)):
        cfg = make_cfg('navier-stokes', order, precision=precision)
        integ = get_integrator(AMDBackend(cfg),
                               BoxMesh((5, 4, 3), warp=_offset), cfg)
        e = integ.system.ele_map['hex']
        assert e.linoff == 0
        # (18, ndims, neles), as the kernel reads them
        c = e._fnorms_linear._host.astype(e._fnorms_linear.dtype)
        c = c.astype(float).reshape(6, 3, 3, e.neles)
        x = HexShape(order).x1d
        xy = np.array([(1, a, b) for b in x for a in x])
        got = np.einsum('pi,fice->fpec', xy, c)
        ref = e._pnorm_fpts.reshape(got.shape)
        mag = np.sqrt((ref**2).sum(axis=-1))
        assert mag.min() > 0.3
        assert (np.abs(got - ref).max(axis=-1)/mag).max() < eps


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['single', 'mixed'])
def test_low_reynolds_away_from_the_origin(backend_factory, precision):
    """Where the viscous terms are large and vertices have few digits left,
    the one-pass kernels are as close to the FP64 run as those they
    replace, which take the stored normals."""
    def step(prec, fuse):
        be = backend_factory(precision=prec, fuse_flux=fuse)
        cfg = make_cfg('navier-stokes', 3, precision=prec, scheme='rk45',
                       dt=1e-3)
        cfg.set('constants', 'mu', '0.1')
        for k, v in (('u', '0.2*sin(y) + 0.1*sin(x)*cos(y)*cos(z)'),
                     ('v', '-0.1*cos(x)*sin(y)*cos(z)'), ('w', '0.1*sin(x)'),
                     ('p', '1/1.4 + 0.02*(cos(2*x) + cos(2*y))')):
            cfg.set('soln-ics', k, v)
        integ = get_integrator(be, BoxMesh(8, warp=lambda x, y, z: (
            x + 100.0 + 0.08*np.sin(y)*np.sin(z), y + 0.05*np.sin(x), z)),
            cfg)
        integ.run_steps(1, 1e-3)
        if prec != 'double':
            assert integ.system._nfv == fuse
        return integ.soln[0].astype(float)
    print(f'\n[hexline low Re] {precision}', flush=True)
    ref = step('double', False)
    sep, one = (rel_l2(step(precision, f), ref) for f in (False, True))
    print(f'[hexline low Re] separate {sep:.2e} one pass {one:.2e}',
          flush=True)
    assert one < 1.1*sep


def test_normals_match_is_checked():
    """A periodic pair of faces whose vertices differ beyond rounding keeps
    the gradients at its interfaces."""
    from pyfr_amd.solvers import NavierStokesIntInters
    m = BoxMesh(2)
    el = _Faces(m, 2)
    i = NavierStokesIntInters.__new__(NavierStokesIntInters)
    from pyfr_amd.solvers import Interside
    i.lhs, i.rhs = (Interside(s) for s in m.con)
    i.elemap, i._perm = {'hex': el}, Ellipsis
    assert i.normals_match
    # vertex 0 of element 0 (x = 0 side) moved by 1e-8
    m.spts['hex'][0, 0, 1] += 1e-8
    i.elemap = {'hex': _Faces(m, 2)}
    del i.__dict__['normals_match']
    assert not i.normals_match


class _Faces:
    """The parts of an element type that its interfaces' normals need."""

    def __init__(self, mesh, order):
        from pyfr_amd.solvers import FluidElements
        cfg = make_cfg('euler', order)
        e = FluidElements(HexShape, mesh.spts['hex'], cfg)
        self.nfacefpts = e.nfacefpts
        self.get_pnorms_for_inters = e.get_pnorms_for_inters


def _hex_args(be, order, neles):
    """Operands of the two entry points for neles elements, every one of
    them padded to a whole block of 64."""
    sh = HexShape(order)
    rng = np.random.default_rng(1)
    m = {k: be.matrix((r, 5, neles), 1 + rng.random((r, 5, neles)),
                      tags={'align'})
         for k, r in (('u', sh.nupts), ('f', sh.nfpts), ('c', sh.nupts),
                      ('g', 3*sh.nfpts))}
    m['s'] = be.matrix((3, sh.nupts, 3, neles),
                       rng.random((3, sh.nupts, 3, neles)), tags={'align'})
    m['r'] = be.matrix((sh.nupts, neles), 1 + rng.random((sh.nupts, neles)),
                       tags={'align'})
    return sh, m


@pytest.mark.gpu
@pytest.mark.parametrize('precision', ['double', 'single'])
@pytest.mark.parametrize('order,neles', [(2, 1), (2, 65), (4, 100)])
def test_short_metric_rows_are_refused(backend_factory, precision, order,
                                       neles):
    """1/|J| rows that do not cover the last block, which every lane of it
    reads.  (The arrays themselves do: nothing here reads past them.)"""
    import ctypes as ct
    from pyfr_amd._lib import FrHipError
    from pyfr_amd.backend import HexLineProvider
    be = backend_factory(precision=precision)
    sh, m = _hex_args(be, order, neles)
    hp = next(p for p in be._providers if isinstance(p, HexLineProvider))
    plan = hp._plan(sh, be.fpdtype)
    u, f, c, g, s, r = (m[k] for k in 'ufcgsr')
    consts = (ct.c_double*8)(1.4, 1e-3, 0.7, 0, 0, 0, 1, 0)

    def div(ldr):
        be.lib.hex_div(plan, 0, neles, u.data, u.leaddim, s.data, s.leaddim,
                       f.data, f.leaddim, c.data, c.leaddim, 1, r.data, ldr,
                       None, 0.0, 0.0, 0, 0, 1.4, None, be.stream)

    def ns(ldr):
        be.lib.hex_nsvol(plan, 0, neles, u.data, u.leaddim, f.data,
                         f.leaddim, s.data, s.leaddim, r.data, ldr, c.data,
                         c.leaddim, g.data, g.leaddim, 0, None, consts, None,
                         be.stream)
    print(f'\n[hexline ldr] {precision} p={order} {neles}', flush=True)
    for call in (div, ns):
        for ldr in (neles, r.leaddim - 1):
            with pytest.raises(FrHipError, match='leading dimensions'):
                call(ldr)
        call(r.leaddim)
    be.wait()
    assert np.isfinite(c.get()).all() and np.isfinite(g.get()).all()
    if precision == 'single':
        # the normal viscous flux in FP32 takes the faces' normals
        with pytest.raises(FrHipError, match='normals'):
            be.lib.hex_nsvol(plan, 1, neles, u.data, u.leaddim, f.data,
                             f.leaddim, s.data, s.leaddim, None, 0, c.data,
                             c.leaddim, g.data, g.leaddim, 1, None, consts,
                             None, be.stream)


@pytest.mark.parametrize('order,neles', [(2, 1), (4, 100)])
def test_unaligned_metric_is_refused(monkeypatch, order, neles):
    """The same at the kernel providers, on the host."""
    import pyfr_amd._lib as _lib
    from pyfr_amd.backend import AMDBackend
    from tests.test_ns_options import StubLib
    monkeypatch.setattr(_lib, '_lib', StubLib())
    be = AMDBackend(make_cfg('navier-stokes', order))
    sh, m = _hex_args(be, order, neles)
    short = be.matrix((sh.nupts, neles))
    tpl = {'c': {'gamma': 1.4}}

    def div(r):
        be.kernel('hexdiv', sh, 0, neles, m['u'], m['f'], m['c'], r, 1.4,
                  m['s'])

    def ns(r):
        be.kernel('hexns', sh, 0, neles, m['u'], m['f'], m['c'], m['g'], tpl,
                  m['s'], r)
    for make in (div, ns):
        make(m['r'])
        with pytest.raises(ValueError, match='Incompatible'):
            make(short)
