"""An infinite element reaches the outputs that depend on it and no others,
though the kernels give absent terms a weight of zero (on the host)."""
import pytest

from cpu_library import run

SPREAD = """
def spread(call, v, k):
    '''outputs that are not finite with v[k] infinite, though they do not depend on v[k]'''
    v = np.array(v)
    a = call(v)
    v[k] += 1.0
    b = call(v)
    v[k] = np.inf
    return int((~np.isfinite(call(v)) & (a == b)).sum())
"""


def test_adjoint_pandya():
    """222_ph: terms the operator does not hold add nothing to its first element"""
    run(SPREAD + """
B = Basis.ho(2, 1)
ctx = E.Context(B)
P, v = ctx.op(-1, random_operator(B, -1, 4)), random_operator(B, 1, 3)
call = lambda x: ctx.commutator_adjoint(P, ctx.op(1, x), 1, mask=E.T222PH).download()
ks = np.flatnonzero(v)[::97][[2, 6, 7, 8, 9]]  # whose terms have no vanishing 6j symbols
assert [spread(call, v, k) for k in ks] == [0] * 5
""")


@pytest.mark.parametrize("rank,dpar", [(2, 0), (2, 2), (4, 0)])
def test_tensor_one_body_terms(rank, dpar):
    """122: at emax 1 every orbit stands alone in its class, so an element of T
    reaches one output; 212 reads T's one-body part only"""
    run(f"""
B = Basis.ho(1, 1)
ctx = E.Context(B)
G, T, R = ctx.op(-1, random_operator(B, -1, 7)), ctx.tensor({rank}, {dpar}), ctx.tensor({rank}, {dpar})
rng = np.random.default_rng(0)
v0 = 1 + len(B.holes) ** 2 + len(B.parts) ** 2 + len(B.parts) * len(B.holes)
for k in rng.choice(np.arange(v0, T.neq), 12, replace=False):
    t = rng.uniform(-1, 1, T.neq)
    t[k] = np.inf
    T.upload(t)
    n = []
    for mask in (8, 16):
        R.clear()
        n.append(int((~np.isfinite(ctx.tensor_commutator(G, T, R, mask=mask).download())).sum()))
    assert n[0] <= 1 and n[1] == 0, (k, n)
""")
