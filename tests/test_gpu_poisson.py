"""The HIP Poisson solver (poisson.hip) against the transform form
(electrostatic/fft.py:9-78 through torch.fft) on random charge densities.

Both are sums of at most 512 terms per axis in FP64: the difference is bounded by
a few hundred roundings of the largest field (1e-12 of it)."""
import ctypes
import types

import pytest
import torch

from bolt_amd import _lib
from bolt_amd.fields import fields_solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2", [(1, 1), (2, 1), (3, 1), (96, 1), (1, 65), (4096, 1), (2, 2),
                                   (3, 4), (32, 32), (5, 512), (511, 7), (33, 50), (128, 96), (256, 256)])
@pytest.mark.parametrize("S", [1, 2])
def test_poisson_matches_the_transforms(gpu, n1, n2, S):
    lib = _lib.load()
    g = _lib.Grid(n1, n2, 4, 4, 1, 1, 0, 0.7 / n1, 1.3 / n2, 1.0, 1.0, 1.0, -2.0, -2.0, -0.5)
    gen = torch.Generator(device="cuda").manual_seed(n1 + 7 * n2)
    Q, eps = n1 * n2, 1.7
    moms = [1.0 + 0.1 * torch.randn(Q, generator=gen, device="cuda", dtype=torch.float64)
            for _ in range(S)]
    charge = [-1.0, 0.6][:S]
    n = lib.boltx_poisson_workspace_size(ctypes.byref(g))
    assert n > 0
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    cc = torch.full((6, Q), float("nan"), device="cuda", dtype=torch.float64)
    st = _lib.stream_handle()
    _lib.check(lib.boltx_poisson_init(ctypes.byref(g), _lib.ptr(ws), st))
    ptrs = (ctypes.c_void_p * S)(*[m.data_ptr() for m in moms])
    _lib.check(lib.boltx_poisson(ctypes.byref(g), S, ptrs, (ctypes.c_double * S)(*charge), eps,
                                 _lib.ptr(cc), _lib.ptr(ws), st))
    ref = torch.zeros(2, Q, device="cuda", dtype=torch.float64)
    fs = types.SimpleNamespace(
        _solver=types.SimpleNamespace(N_q1=n1, N_q2=n2), dq1=0.7 / n1, dq2=1.3 / n2,
        params=types.SimpleNamespace(eps=eps))
    fields_solver._poisson(fs, sum(c * m for c, m in zip(charge, moms)), ref)
    err = (cc[:2] - ref).abs().max().item()
    assert err <= 1e-12 * max(ref.abs().max().item(), 1e-3), err
    assert torch.isnan(cc[2:]).all()  # rows 2-5 are not the solver's


def test_poisson_sizes_it_does_not_take():
    lib = _lib.load()
    for n1, n2 in ((4097, 1), (513, 2), (2, 513), (512, 512)):
        g = _lib.Grid(n1, n2, 4, 4, 1, 1, 0, 0.1, 0.1, 1.0, 1.0, 1.0, -2.0, -2.0, -0.5)
        assert lib.boltx_poisson_workspace_size(ctypes.byref(g)) == 0
        assert lib.boltx_poisson_init(ctypes.byref(g), ctypes.c_void_p(16), None) == -3
