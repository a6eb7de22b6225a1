"""Whole steps in one library call (boltx_advance) against the same step issued
stage by stage: the same arithmetic, so the states are equal bit for bit, and
so are the steps that raise the divergence flag."""
import ctypes

import pytest
import torch

from bolt_amd import _lib
from tests.cases import case_2d2v, case_bc, case_c1, case_es, case_species, hip_solver

pytestmark = pytest.mark.gpu

CASES = {
    "1d1v": lambda st: case_c1(seed=1, stepper=st),
    "lines fp64": lambda st: case_2d2v(seed=2, N_q=64, N_p=9, stepper=st),
    "lines fp32": lambda st: case_2d2v(seed=2, N_q=64, N_p=11, stepper=st,
                                       precision="fp32-bulk"),
    "mirror": lambda st: case_bc(stepper=st, left="mirror", right="mirror", bottom="mirror",
                                 top="mirror"),
    "electrostatic": lambda st: case_es(seed=4, N_q1=16, N_q2=12, N_p=10, stepper=st),
    "two species": lambda st: case_species(N_q1=64, memory_layout="q1-lines", stepper=st),
    "two species es": lambda st: case_species(
        masses=(1.0, 25.0), charges=(-1.0, 1.0), p_max=(6.0, 1.5), N_q1=32, N_q2=1, N_p1=16,
        N_p2=1, p_dim=1, fields=True, fields_type="electrostatic", stepper=st),
}


@pytest.mark.parametrize("stepper", ["RK2", "SSP-RK3"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_whole_step_equals_its_stages(gpu, name, stepper):
    c = CASES[name](stepper)
    a, b = hip_solver(c), hip_solver(c)
    for _ in range(3):
        a.strang_timestep(c.dt)
        b._stage_events = []  # timed stages are issued one by one
        b.strang_timestep(c.dt)
    assert b._stage_events
    for x, y in zip(a._spc, b._spc):
        assert torch.equal(x.f, y.f) and torch.equal(x.mom, y.mom)
    assert a.time_elapsed == b.time_elapsed
    if a.fields_solver is not None:
        assert a.fields_solver.at_n == b.fields_solver.at_n
        assert torch.equal(a.fields_solver._cc, b.fields_solver._cc)
    a._spc[-1].f.view(-1)[7] = float("nan")
    a._advance(c.dt)
    with pytest.raises(SystemExit):
        a.check_divergence()


def test_a_dirichlet_side_is_refused(gpu):
    s = hip_solver(case_bc(left="dirichlet"))
    x = _lib.State(ctypes.pointer(s._grid), ctypes.pointer(s._phys), *[
        s._f.data_ptr(), s._buf("u1").data_ptr(), s._buf("u2").data_ptr(), s._mom.data_ptr(),
        s._mom.clone().data_ptr(), s._mom.clone().data_ptr(),
        0 if s._ws is None else s._ws.data_ptr()])
    f = s._f.clone()
    rc = s._L.boltx_advance(1, ctypes.byref(x), 0, 1e-3, 1.0, None, None, None,
                            _lib.stream_handle())
    assert rc == -3 and torch.equal(f, s._f)
