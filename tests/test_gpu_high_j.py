"""Many orbits of which a few have 2j = 29: their Pandya columns stage more than
64 KiB of tables while the two-body part (2.7e6 elements) is small enough for
the merged commutator.  Against the separate kernels, which run while
profiling is on: the same bits."""
import numpy as np
import pytest

from imsrg_mi355x import Basis, random_operator

pytestmark = pytest.mark.gpu


def test_high_j_merged():
    from imsrg_mi355x import engine as E
    low = [(0, 1), (1, 1), (1, 3), (2, 3), (2, 5), (3, 5), (3, 7)]
    orb = [o for tz in (-1, 1) for o in [(k, l, j, tz) for l, j in low for k in range(5)] +
           [(k, 14, 29, tz) for k in range(3)]]
    B = Basis.from_orbits(orb, [int(o[0] == 0 and o[1] == 0) for o in orb])
    ctx = E.Context(B)
    ctx.set_tile_shapes(0, 0)
    L, R = ctx.op(-1, random_operator(B, -1, 1)), ctx.op(1, random_operator(B, 1, 2))
    got = ctx.commutator(L, R).download()
    ctx.profile(True)
    want = ctx.commutator(L, R).download()
    assert ctx.profile_read()["gemm_pphh"][1] == 1
    assert np.linalg.norm(got) > 0 and np.array_equal(got, want)
