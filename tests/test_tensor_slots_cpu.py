"""The slot lists of the tensor recoupling and Pandya kernels on the host, every
read checked: ranks for which some class's scan, after batches of exactly 32
slots, ends without another (rank 4 and 10 at emax 3; none at rank 2)."""
import pytest

from cpu_library import run

CODE = """
B = Basis.ho(%d, 1)
ctx = E.Context(B)
T = ctx.tensor(%d, %d, 1)
T.upload(np.random.default_rng(1).uniform(-1, 1, T.neq))
r = ctx.tensor_commutator(ctx.op(-1, 1e-2 * random_operator(B, -1, 1)), T).download()
assert np.isfinite(r).all() and np.linalg.norm(r) > 0
"""


@pytest.mark.parametrize("emax,rank,dpar", [(1, 2, 2), (3, 2, 0), (3, 4, 0), (3, 4, 2), (3, 10, 0)])
def test_empty_batches(emax, rank, dpar):
    run(CODE % (emax, rank, dpar))
