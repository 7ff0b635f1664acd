"""The five-launch commutator against the separate kernels.

Both make every sum in the same order, so results are equal bit for bit; the
separate kernels run while profiling is on.  Bases on both sides of the lines
where its first launch splits up (10^6 and, for one instance, 3 10^6 two-body
elements), with unequal proton and neutron holes and instances that one series
drops early."""
import numpy as np
import pytest

from imsrg_mi355x import Basis, random_operator
from imsrg_mi355x.basis import closed_shell_con, hk_orbits

pytestmark = pytest.mark.gpu


def basis(emax, kp, kn):
    orb = hk_orbits(emax)
    cp, cn = closed_shell_con(orb, kp), closed_shell_con(orb, kn)
    return Basis.from_orbits(orb, [p if o[3] < 0 else n for o, p, n in zip(orb, cp, cn)])


@pytest.mark.parametrize("emax,kp,kn,nb", [(3, 1, 3, 15), (4, 3, 1, 17), (5, 1, 6, 1), (6, 6, 1, 2), (7, 3, 1, 1),
                                           (8, 1, 1, 1)])
def test_merged_bits(emax, kp, kn, nb):
    from imsrg_mi355x import engine as E
    B = basis(emax, kp, kn)
    ctx = E.Context(B, nbatch=nb)
    ctx.set_tile_shapes(0, 0)
    assert ctx.info()["vsize"] * nb > 2e5
    G = ctx.op(-1, np.stack([random_operator(B, -1, 10 + k) for k in range(nb)]))
    H = ctx.op(1, np.stack([random_operator(B, 1, 20 + k) * 10.0 ** -(k % 5) for k in range(nb)]))
    G.scale(1e-3)
    got, (HS, n) = ctx.commutator(G, H).download(), ctx.bch(G, H)
    ctx.profile(True)
    want, (HW, m) = ctx.commutator(G, H).download(), ctx.bch(G, H)
    assert ctx.profile_read()["gemm_pphh"][1] > 1
    assert np.array_equal(got, want)
    assert np.array_equal(n, m) and np.array_equal(HS.download(), HW.download())
