"""The marching stages (psplit.h), two kernels with three p axes and one without
p-advection, and the currents the first forms, against the generic kernel on
random states.

Both evaluate the same formulas; FP64 differs by rounding (the per-RHS bar of
the parity tests, 1e-12), FP32 by a few roundings of each term (1e-6)."""
import ctypes

import pytest
import torch

from bolt_amd import _lib
from tests.cases import case_2d2v, case_2d3v, hip_solver

pytestmark = pytest.mark.gpu


def _solver(nq, np_, recon, precision, walls=False):
    c = case_2d3v(seed=3, N_q=8, N_p=4, N_q1=nq[0], N_q2=nq[1], N_p1=np_[0], N_p2=np_[1],
                  N_p3=np_[2], recon_q=recon[0], recon_p=recon[1], precision=precision)
    if walls:
        c.params.fields_type, c.params.fields_initialize = "electrostatic", "fft"
        c.params.fields_solver = "fft"
        bc = c.boundary_conditions
        bc.in_q1_left = bc.in_q1_right = bc.in_q2_bottom = bc.in_q2_top = "mirror"
    return hip_solver(c)


def _random_stage(s, seed, form):
    g = torch.Generator(device=s.device).manual_seed(seed)

    def rand(shape, dtype=torch.float64):
        return torch.rand(shape, generator=g, device=s.device, dtype=torch.float64).to(dtype)

    # where the marching stages apply: these are the workspaces with room for them
    assert s._ws.numel() > 16 * s._P + 4096
    u, un, w = (s._alloc_f() for _ in range(3))
    for x in (u, un, w):
        x.copy_(0.5 + rand(x.shape, x.dtype))
    s._fill_ghosts(u)
    mom = torch.empty_like(s._mom)
    _lib.check(s._L.boltx_moments(ctypes.byref(s._grid), ctypes.byref(s._phys), _lib.ptr(u),
                                  _lib.ptr(mom), _lib.ptr(s._ws), _lib.stream_handle()))
    F = [rand((6, s._Q)) - 0.5 for _ in range(3)]
    a, b, w = {"first": (0.0, 1.0, u), "combine": (0.75, 0.25, u), "midpoint": (0.0, 1.0, w),
               "general": (0.3, 0.7, w)}[form]
    return u, w, un, mom, F, a, b


def _run(s, entry, inputs, ws, currents):
    u, w, un, mom, F, a, b = inputs
    out = s._alloc_f()
    out.fill_(float("nan"))
    mo = torch.full_like(mom, float("nan"))
    J = torch.full((3, s._Q), float("nan"), device=s.device, dtype=torch.float64)
    st = _lib.Stage(_lib.ptr(u), _lib.ptr(w), _lib.ptr(un), _lib.ptr(out), a, b, 1e-3,
                    _lib.ptr(mom), _lib.ptr(mo), *[_lib.ptr(x) for x in F], _lib.ptr(ws),
                    _lib.ptr(J) if currents else None)
    _lib.check(getattr(s._L, entry)(ctypes.byref(s._grid), ctypes.byref(s._phys),
                                    ctypes.byref(st), _lib.stream_handle()))
    return out, mo[:5], J


def _close(a, b, tol):
    assert torch.isfinite(a).all()
    err = ((a.double() - b.double()).abs().max() / b.double().abs().max()).item()
    assert err <= tol, err


@pytest.mark.parametrize("nq,np_,recon,form", [
    ((205, 486), (2, 2, 2), ("weno5", "weno5"), "first"),
    ((89, 85), (3, 5, 7), ("ppm", "weno5"), "combine"),
    ((16, 19), (24, 24, 5), ("ppm", "weno5"), "general"),
    ((401, 1), (26, 26, 3), ("minmod", "ppm"), "combine"),
    ((31, 33), (13, 5, 12), ("piecewise-constant", "minmod"), "first"),
    ((45, 47), (8, 8, 6), ("ppm", "piecewise-constant"), "general"),
    ((31, 32), (9, 7, 13), ("minmod", "weno5"), "midpoint"),
])
@pytest.mark.parametrize("precision", ["fp64", "fp32-bulk"])
def test_split_stage_matches_the_generic_kernel(gpu, nq, np_, recon, form, precision):
    s = _solver(nq, np_, recon, precision)
    x = _random_stage(s, 7, form)
    ref = _run(s, "boltx_fvm_stage", x, None, True)
    got = _run(s, "boltx_fvm_stage", x, s._ws, True)
    tol = 1e-12 if precision == "fp64" else 1e-6
    for r, o in zip(ref, got):
        _close(o, r, tol)
    # the currents alone, with and without the workspace
    J = torch.full_like(ref[2], float("nan"))
    _lib.check(s._L.boltx_currents_ws(ctypes.byref(s._grid), ctypes.byref(s._phys),
                                      _lib.ptr(x[0]), _lib.ptr(J), _lib.ptr(s._ws),
                                      _lib.stream_handle()))
    _close(J, ref[2], tol)
    # the stage that takes the q-fluxes of that call: the same bits
    for a, b in zip(got[:2], _run(s, "boltx_fvm_stage_after_currents", x, s._ws, False)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32-bulk"])
def test_split_stage_with_ghost_rows(gpu, precision):
    s = _solver((83, 80), (6, 4, 5), ("weno5", "minmod"), precision, walls=True)
    x = _random_stage(s, 8, "combine")
    ref = _run(s, "boltx_fvm_stage", x, None, False)
    got = _run(s, "boltx_fvm_stage", x, s._ws, False)
    for r, o in zip(ref[:2], got[:2]):
        _close(o, r, 1e-12 if precision == "fp64" else 1e-6)


@pytest.mark.parametrize("precision,nq", [("fp64", 32), ("fp32-bulk", 46)])
def test_split_stage_in_chunks_is_bitwise_the_same(gpu, precision, nq):
    """boltx_fvm_stage_noalloc works in q2 chunks that its scratch array
    holds (here two), boltx_fvm_stage in one."""
    s = _solver((nq, nq), (20, 20, 20), ("ppm", "weno5"), precision)
    assert s._f.numel() * s._f.element_size() > 40 << 20
    x = _random_stage(s, 9, "combine")
    for a, b in zip(_run(s, "boltx_fvm_stage", x, s._ws, True),
                    _run(s, "boltx_fvm_stage_noalloc", x, None, True)):
        assert torch.equal(a, b)


def _fields_off(nq, np_, recon, precision, walls=""):
    c = case_2d2v(seed=5, N_q=8, N_p=4, N_q1=nq[0], N_q2=nq[1], N_p1=np_[0], N_p2=np_[1],
                  N_p3=np_[2], recon_q=recon, precision=precision, memory_layout="reference",
                  p_dim=sum(n > 1 for n in np_))
    bc = c.boundary_conditions
    if "1" in walls:
        bc.in_q1_left = bc.in_q1_right = "mirror"
    if "2" in walls:
        bc.in_q2_bottom = bc.in_q2_top = "mirror"
    return hip_solver(c)


@pytest.mark.parametrize("nq,np_,recon,form,walls", [
    ((101, 75), (30, 28, 1), "ppm", "combine", ""),
    ((64, 67), (24, 24, 1), "weno5", "first", ""),
    ((3, 5), (500, 600, 1), "minmod", "midpoint", ""),
    ((2051, 1), (32, 65, 1), "piecewise-constant", "general", ""),
    ((33, 34), (12, 11, 13), "ppm", "general", ""),
    ((50, 47), (27, 27, 1), "weno5", "combine", "1"),
    ((93, 95), (27, 27, 1), "ppm", "first", "2"),
    ((45, 51), (30, 26, 1), "weno5", "midpoint", "12"),
])
@pytest.mark.parametrize("precision", ["fp64", "fp32-bulk"])
def test_marching_stage_matches_the_generic_kernel(gpu, nq, np_, recon, form, walls, precision):
    if precision != "fp64" and recon == "weno5":
        pytest.skip("FP32 WENO5 keeps the slab kernel")
    s = _fields_off(nq, np_, recon, precision, walls)
    x = _random_stage(s, 11, form)
    for r, o in zip(_run(s, "boltx_fvm_stage", x, None, False)[:2],
                    _run(s, "boltx_fvm_stage", x, s._ws, False)[:2]):
        _close(o, r, 1e-12 if precision == "fp64" else 1e-6)


def test_marching_stage_in_chunks_is_bitwise_the_same(gpu):
    s = _fields_off((300, 200), (16, 16, 1), "ppm", "fp64")
    need = 300 * 200 * (33 * 8 + 4 * 5 * 8)
    s2 = _fields_off((900, 200), (16, 16, 1), "ppm", "fp64")
    for sv, chunks in ((s, need > 40 << 20), (s2, 3 * need > 40 << 20)):
        x = _random_stage(sv, 12, "combine")
        for a, b in zip(_run(sv, "boltx_fvm_stage", x, sv._ws, False)[:2],
                        _run(sv, "boltx_fvm_stage_noalloc", x, None, False)[:2]):
            assert torch.equal(a, b)
    assert chunks
