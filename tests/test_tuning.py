"""Which callers of the flux-folded divergence the tuner times for: plain
right-hand sides and RK4 stages each keep a variant of their own."""
import numpy as np
import pytest

import pyfr_amd._lib as _lib
from pyfr_amd.backend import AMDBackend, MulProvider
from pyfr_amd.cases import make_simplex_cfg
from pyfr_amd.mesh import SimplexBoxMesh
from pyfr_amd.solvers import get_integrator
from tests.test_ns_options import StubLib


class _Recorder(StubLib):
    def __init__(self):
        super().__init__()
        self.tuned = []

    def __getattr__(self, name):
        fn = super().__getattr__(name)
        if name == 'tdivf_plan_create':
            def create(ref, *args):
                # a handle of its own for each plan
                self._next += 64
                ref._obj.value = self._next
            return create
        if name.startswith('tdivf_plan_tune'):
            def note(plan, *args):
                self.tuned.append(name)
                fn(plan, *args)
            return note
        return fn


def _integ(be, scheme, precision='single'):
    cfg = make_simplex_cfg(3, precision=precision, scheme=scheme)
    be = be or AMDBackend(cfg)
    return get_integrator(be, SimplexBoxMesh.stacked(2, 1, 1), cfg)


@pytest.mark.parametrize('scheme,calls,names', [
    ('rk4', 'rhs', {'tdivf_plan_tune'}),
    ('rk4', 'step', {'tdivf_plan_tune_rk4'}),
    ('rk45', 'step', {'tdivf_plan_tune'}),
    ('rk4', 'rhs step', {'tdivf_plan_tune', 'tdivf_plan_tune_rk4'})])
def test_each_caller_tunes_its_own(monkeypatch, scheme, calls, names):
    lib = _Recorder()
    monkeypatch.setattr(_lib, '_lib', lib)
    integ = _integ(None, scheme)
    for _ in range(2):
        if 'rhs' in calls:
            integ.system.rhs(0.0, 0, 1)
        if 'step' in calls:
            integ.run_steps(1, 1e-3)
    # each once for the tets and once for the prisms
    assert sorted(lib.tuned) == sorted(2*list(names))


@pytest.mark.gpu
def test_rk4_tuning_leaves_right_hand_sides_alone(backend_factory):
    """The 16-row tiles forced on a plan serve right-hand sides before and
    after RK4 stages choose theirs; both report what they run."""
    be = backend_factory(precision='single', graphs=False)
    integ = _integ(be, 'rk4')
    sysm = integ.system
    sysm.rhs(0.0, 0, 1)
    mp = next(p for p in be._providers if isinstance(p, MulProvider))
    for plan, _, _ in mp._plans3.values():
        be.lib.tdivf_plan_set_variant(plan, 4)
    sysm.rhs(0.0, 0, 1)
    before = sysm.ele_scal_upts(1)
    assert sysm.fused_rk4
    sysm.rhs(0.0, 0, 1)
    for a, b in zip(before, sysm.ele_scal_upts(1)):
        assert np.array_equal(a, b)
    kinds = sorted(t['kernel'] for t in mp.tuning_report()
                   if t['kernel'].startswith('tdivf'))
    assert kinds == 2*['tdivf_flux'] + 2*['tdivf_flux_rk4']
