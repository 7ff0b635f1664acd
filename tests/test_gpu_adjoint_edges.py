"""The adjoint commutator in bases whose blocks end inside its 32 x 32 tiles:
<C, [P, Y]> = <Ybar, Y> (Frobenius products over the full layout), to 1e-11 of
the largest partial sum, for odd sizes and unequal proton and neutron holes."""
import numpy as np
import pytest

from imsrg_mi355x import random_operator
from test_gpu_adjoint import frob
from test_gpu_small_path import basis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hP,hY", [(-1, 1), (1, -1)])
@pytest.mark.parametrize("emax,kp,kn", [(1, 1, 1), (2, 3, 1), (3, 1, 6), (5, 3, 6)])
def test_adjoint_identity_odd_bases(emax, kp, kn, hP, hY):
    from imsrg_mi355x import engine as E
    B, hC = basis(emax, kp, kn), -hP * hY
    ctx = E.Context(B)
    P, Y, Cb = random_operator(B, hP, 31), random_operator(B, hY, 32), random_operator(B, hC, 33)
    Cb[0] = 0.7
    dP, dY, dC = ctx.op(hP, P), ctx.op(hY, Y), ctx.op(hC, Cb)
    lhs = frob(B, Cb, hC, ctx.commutator(dP, dY).download(), hC)
    yb = ctx.commutator_adjoint(dP, dC, hY).download()
    rhs = frob(B, yb, hY, Y, hY)
    scale = np.linalg.norm(yb) * np.linalg.norm(Y)
    assert abs(lhs - rhs) <= 1e-11 * scale
