"""Dynamic LDS past 64 KiB has to be allowed for a kernel before its launch; on
the host such a launch fails otherwise (the kernels themselves are not run
here).  Bases of many orbits of which a few have 2j = 29 stage more than that for
their Pandya columns, though their two-body part is that of a merged
commutator."""
from cpu_library import run

HIGH_J = """
low = [(0, 1), (1, 1), (1, 3), (2, 3), (2, 5), (3, 5), (3, 7)]
def basis(nj):
    orb = [o for tz in (-1, 1) for o in [(k, l, j, tz) for l, j in low for k in range(5)] + [(k, 14, 29, tz) for k in range(nj)]]
    return Basis.from_orbits(orb, [int(o[0] == 0 and o[1] == 0) for o in orb])
B = basis(3)
ctx = E.Context(B)
"""


def test_high_j_commutator():
    run(HIGH_J + "ctx.commutator(ctx.op(-1), ctx.op(1))", IMSRG_EMU_CHECK=1)


def test_second_context_keeps_the_limit():
    """a later context of a smaller basis, still past 64 KiB, takes nothing back"""
    run(HIGH_J + """
B2 = basis(5)
big = E.Context(B2)
ctx = E.Context(B)
big.commutator_adjoint(big.op(-1), big.op(1), 1)
big.cross_coupled(big.op(1))
""", IMSRG_EMU_CHECK=1)


def test_second_tensor_space_keeps_the_limit():
    """E1, then E2, in one context: the one-body kernel of the first still starts"""
    run("""
ctx = E.Context(Basis.ho(5, 1))
E1, E2, G = ctx.tensor(2, 2), ctx.tensor(4, 0), ctx.op(-1)
ctx.tensor_commutator(G, E1)
ctx.tensor_commutator(G, E2)
""", IMSRG_EMU_CHECK=1)
