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
