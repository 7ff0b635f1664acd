"""Series gates made in the next commutator's first launch (small bases).

Against the separate kernels, which run while profiling is on and keep a launch
for every gate: term counts and results are equal, bit for bit, when the instances
of a batch stop at different terms, at once, or never (the clipping error); a
series that ends leaves nothing for the next call."""
import numpy as np
import pytest

from imsrg_mi355x import Basis, random_operator

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,scales", [(1, [3e-3]), (2, [1e-2, 0.0, 1e-5, 3e-3]), (3, [2e-3, 1e-6, 1e-4]), (4, [0.0, 1e-3])])
def test_gates_in_batches(emax, scales):
    from imsrg_mi355x import engine as E
    B, nb = Basis.ho(emax, 1), len(scales)
    ctx = E.Context(B, nbatch=nb)
    assert ctx.info()["vsize"] * nb <= 2e5
    G = ctx.op(-1, np.stack([x * random_operator(B, -1, 10 + k) for k, x in enumerate(scales)]))
    H = ctx.op(1, np.stack([random_operator(B, 1, 20 + k) for k in range(nb)]))
    D = np.stack([random_operator(B, -1, 30 + k) for k in range(nb)])
    out = []
    for prof in (False, True):
        ctx.profile(prof)
        HS, n = ctx.bch(G, H)
        DG, m = ctx.magnus_expand(ctx.op(-1, D), G)
        C = ctx.commutator(G, H)
        out.append((np.atleast_1d(n).tolist(), np.atleast_1d(m).tolist(), HS.download(), DG.download(), C.download()))
    assert out[0][:2] == out[1][:2]
    assert all(np.array_equal(a, b) for a, b in zip(out[0][2:], out[1][2:]))


def test_clipped_series_leaves_nothing():
    from imsrg_mi355x import engine as E
    B = Basis.ho(2, 1)
    ctx = E.Context(B)
    G, H = ctx.op(-1, random_operator(B, -1, 1)), ctx.op(1, random_operator(B, 1, 2))
    want = ctx.commutator(G, H).download()
    G.scale(1e3)
    with pytest.raises(Exception, match="clipping BCH"):
        ctx.bch(G, H)
    G.scale(1e-3)
    got = ctx.commutator(G, H).download()
    # the scaling back and forth rounds each element of G twice
    assert np.allclose(got, want, rtol=0, atol=1e-13 * np.abs(want).max() * B.nsp)
    G.scale(1e-2)
    out = []
    for prof in (False, True):
        ctx.profile(prof)
        HS, n = ctx.bch(G, H)
        out.append((n, HS.download()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
