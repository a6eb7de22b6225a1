"""The q1-line march with neighbours from DPP rotates (a line of exactly 1, 2 or
4 cells per lane) against the same stage on arrays one element off that
alignment, which takes the LDS lines, and against the reference-layout kernel.

Both marches evaluate the same explicitly fused expressions: equal bit for bit.
The reference-layout kernel differs by rounding (1e-12 of the largest value)."""
import ctypes

import pytest
import torch

from bolt_amd import _lib
from tests.cases import case_2d2v, hip_solver

pytestmark = pytest.mark.gpu


def _off(x, by):
    """x in storage whose first element is ``by`` elements into an allocation."""
    y = torch.empty(x.numel() + by, dtype=x.dtype, device=x.device)[by:]
    return y.copy_(x.reshape(-1))


def _stage(s, u, w, un, coef, mom, by):
    args = [_off(x, by) for x in (u, w, un, torch.zeros_like(u))]
    if coef[3]:
        args[1] = args[0]  # w is u
    mo = torch.zeros_like(mom)
    st = _lib.Stage(*[_lib.ptr(x) for x in args], *coef[:3], _lib.ptr(mom), _lib.ptr(mo), None,
                    None, None, _lib.ptr(s._ws), None)
    _lib.check(s._L.boltx_fvm_stage(ctypes.byref(s._grid), ctypes.byref(s._phys),
                                    ctypes.byref(st), _lib.stream_handle()))
    torch.cuda.synchronize()
    return args[3].reshape(u.shape).clone(), mo


@pytest.mark.parametrize("coef", [(0.0, 1.0, 1e-3, True), (0.75, 0.25, 1e-3, True),
                                  (0.0, 1.0, 1e-3, False), (0.3, 0.6, 1e-3, False)])
@pytest.mark.parametrize("recon", ["piecewise-constant", "minmod", "ppm", "weno5"])
@pytest.mark.parametrize("n1,n2,precision", [(64, 5, "fp64"), (64, 16, "fp64"), (128, 7, "fp64"),
                                             (128, 1, "fp64"), (256, 6, "fp64"),
                                             (256, 33, "fp32-bulk"), (256, 1, "fp32-bulk")])
def test_rotated_march(gpu, n1, n2, precision, recon, coef):
    def make(layout):
        return hip_solver(case_2d2v(seed=5, N_q1=n1, N_q2=n2, N_p=5, recon_q=recon,
                                    recon_p=recon, precision=precision, memory_layout=layout))
    s = make("q1-lines")
    g = torch.Generator(device=gpu).manual_seed(n1 + n2)
    u, w, un = ((1.0 + 0.3 * torch.rand(s._f.shape, generator=g, device=gpu,
                                        dtype=torch.float64)).to(s._dtype) for _ in range(3))
    mom = s._mom.clone()
    a, ma = _stage(s, u, w, un, coef, mom, 0)
    b, mb = _stage(s, u, w, un, coef, mom, 1)
    assert torch.equal(a, b) and torch.equal(ma, mb)
    if precision == "fp64":
        r = make("reference")
        flip = [x.transpose(1, 2).contiguous() for x in (u, w, un)]
        c, mc = _stage(r, *flip, coef, mom, 0)
        assert (a - c.transpose(1, 2)).abs().max() <= 1e-12 * a.abs().max()
        assert (ma[:5] - mc[:5]).abs().max() <= 1e-12 * mc[:5].abs().max()
