"""Options that a Navier-Stokes run cannot do without, on the host: the
solver is built and its right-hand side's kernels are made with a library
that launches nothing."""
import pytest

import pyfr_amd._lib as _lib
from pyfr_amd.cases import make_cfg, make_simplex_cfg
from pyfr_amd.mesh import BoxMesh, SimplexBoxMesh


class StubLib:
    """Accepts every call; memory is a counter."""

    def __init__(self):
        self._next = 1 << 20

    def malloc(self, ref, nbytes):
        ref._obj.value = self._next
        self._next += (nbytes + 4095)//4096*4096

    def __getattr__(self, name):
        def fn(*args):
            # whatever is handed back by reference: a handle or a kind
            for a in args:
                if hasattr(a, '_obj'):
                    a._obj.value = 2
        return fn


def _run(monkeypatch, kind, drop=None, fuse=True):
    from pyfr_amd.backend import AMDBackend
    from pyfr_amd.solvers import get_integrator
    monkeypatch.setattr(_lib, '_lib', StubLib())
    if kind == 'hex':
        cfg, mesh = make_cfg('navier-stokes', 2, scheme='rk45'), BoxMesh(2)
    else:
        cfg = make_simplex_cfg(2, system='navier-stokes', scheme='rk45')
        mesh = SimplexBoxMesh.stacked(2, 1, 1)
    cfg.set('backend-hip', 'fused', str(fuse))
    if drop is not None:
        assert cfg._cp.remove_option(*drop)
    integ = get_integrator(AMDBackend(cfg), mesh, cfg)
    integ.run_steps(1, 1e-3)


@pytest.mark.parametrize('kind', ['hex', 'simplex'])
@pytest.mark.parametrize('fuse', [True, False])
def test_complete_run(monkeypatch, kind, fuse):
    _run(monkeypatch, kind, fuse=fuse)


@pytest.mark.parametrize('kind', ['hex', 'simplex'])
@pytest.mark.parametrize('fuse', [True, False])
@pytest.mark.parametrize('drop', [('constants', 'mu'), ('constants', 'Pr'),
                                  ('solver-interfaces', 'ldg-tau')])
def test_missing_option_is_refused(monkeypatch, kind, fuse, drop):
    """A run without mu would be inviscid, without a word."""
    with pytest.raises(KeyError, match=drop[1]):
        _run(monkeypatch, kind, drop, fuse)
