"""The two-body transform to the Hartree-Fock basis in wide channel blocks,
where fewer rows are staged per workgroup (more than 1024 and more than 2048
pair states), and in groups of up to seven orbits.

With coefficients that are signs, every output is one product with the weights'
signs plus exact zeros: any signs s give s_a s_b s_c s_d times what the
identity gives, bit for bit, and the identity leaves the elements between
pairs of distinct orbits as they are (a pair of equal orbits has a weight of
two rounded square roots)."""
import numpy as np
import pytest

from imsrg_mi355x import Basis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,shells,wide", [(4, 3, 0), (10, 3, 1024), (12, 1, 2048)])
def test_sign_transform(emax, shells, wide):
    from imsrg_mi355x import engine as E
    B = Basis.ho(emax, shells)
    assert max(b.dim for b in B.blocks) > wide
    rng = np.random.default_rng(emax)
    jj, l, tz = (np.asarray(x).astype(int) for x in (B.jj, B.l, B.tz))
    same = (jj[:, None] == jj) & (l[:, None] == l) & (tz[:, None] == tz)
    f = np.where(same, rng.uniform(-1, 1, same.shape), 0.0)
    vec = rng.uniform(-1, 1, B.neq)
    s = rng.choice([-1.0, 1.0], B.nsp)
    pairs = [np.concatenate(b.pairs) if b.dim else np.zeros((0, 2), int) for b in B.blocks]
    ps = [s[p[:, 0]] * s[p[:, 1]] for p in pairs]
    forbidden = [(p[:, 0] == p[:, 1]) & (b.J // 2 % 2 == 1) for b, p in zip(B.blocks, pairs)]
    mask = [np.outer(~x, ~x).astype(float) for x in forbidden]
    vec *= B.vec_from_full(1.0, np.zeros((B.nsp, B.nsp)), mask)
    vec += B.vec_from_full(0.0, f + f.T, [0.0 * m for m in mask])
    sign = B.vec_from_full(1.0, np.outer(s, s), [np.outer(x, x) for x in ps])
    ctx = E.Context(B)
    eye, flip = (ctx.op(1, vec).to_hf(np.diag(d)).download() for d in (np.ones(B.nsp), s))
    v0 = 1 + len(B.holes) ** 2 + len(B.parts) ** 2 + len(B.parts) * len(B.holes)
    distinct = B.vec_from_full(0.0, np.zeros((B.nsp, B.nsp)),
                               [np.outer(p[:, 0] != p[:, 1], p[:, 0] != p[:, 1]).astype(float) for p in pairs])[v0:] > 0
    assert np.array_equal(eye[v0:][distinct], vec[v0:][distinct])
    assert np.array_equal(flip, sign * eye)
    ctx.close()
