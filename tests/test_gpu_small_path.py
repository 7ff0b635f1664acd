"""The three-launch commutator of small bases against the separate kernels.

Both make every sum in the same order, so results are equal bit for bit; the
separate kernels run while profiling is on.  Bases: the smallest, odd ones with
unequal proton and neutron holes (blocks that end inside a 16 x 16 tile, ph
runs past sixteen terms), the largest the rule takes, and batches."""
import numpy as np
import pytest

from imsrg_mi355x import Basis, random_operator
from imsrg_mi355x.basis import closed_shell_con, hk_orbits

pytestmark = pytest.mark.gpu


def basis(emax, kp, kn):
    orb = hk_orbits(emax)
    cp, cn = closed_shell_con(orb, kp), closed_shell_con(orb, kn)
    return Basis.from_orbits(orb, [p if o[3] < 0 else n for o, p, n in zip(orb, cp, cn)])


@pytest.mark.parametrize("hl,hr", [(-1, 1), (-1, -1), (1, 1)])
@pytest.mark.parametrize("emax,kp,kn,nb", [(1, 1, 1, 1), (2, 1, 3, 5), (3, 3, 1, 3), (4, 3, 6, 1), (5, 6, 3, 1),
                                           (6, 3, 3, 1)])
def test_small_path_bits(emax, kp, kn, nb, hl, hr):
    from imsrg_mi355x import engine as E
    B = basis(emax, kp, kn)
    ctx = E.Context(B, nbatch=nb)
    assert ctx.info()["vsize"] * nb <= 1e6
    L = ctx.op(hl, np.stack([random_operator(B, hl, 10 + k) for k in range(nb)]))
    R = ctx.op(hr, np.stack([random_operator(B, hr, 20 + k) for k in range(nb)]))
    got = ctx.commutator(L, R).download()
    ctx.profile(True)
    want = ctx.commutator(L, R).download()
    assert ctx.profile_read()["gemm_pphh"][1] == 1
    assert np.array_equal(got, want)


def test_small_path_series():
    """BCH and Magnus truncation and sums, both ways: equal term counts and bits"""
    from imsrg_mi355x import engine as E
    B = basis(3, 3, 1)
    ctx = E.Context(B)
    G, H = ctx.op(-1, random_operator(B, -1, 1)), ctx.op(1, random_operator(B, 1, 2))
    G.scale(2e-3)
    out = []
    for prof in (False, True):
        ctx.profile(prof)
        HS, n = ctx.bch(G, H)
        DG, m = ctx.magnus_expand(ctx.op(-1, random_operator(B, -1, 3)), G)
        out.append((HS.download(), n, DG.download(), m))
    assert out[0][1] == out[1][1] > 3 and out[0][3] == out[1][3] > 1
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][2], out[1][2])
