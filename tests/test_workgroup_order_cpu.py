"""Kernels in which one workgroup writes what others of the launch read, on the
host with two workgroups interleaved: one wavefront of the second starts, the
first runs whole, then the rest of the second.  Every wavefront of a workgroup
has to come to the same answer (a barrier that some have left ends the run),
and results do not depend on the order."""
import functools

import pytest

from cpu_library import run

in_order = functools.lru_cache(run)

SERIES = """
B = Basis.ho(1, 1)
ctx = E.Context(B, nbatch=3)
G = ctx.op(-1, np.stack([x * random_operator(B, -1, 10 + k) for k, x in enumerate((1e-2, 0, 1e-3))]))
H = ctx.op(1, np.stack([random_operator(B, 1, 20 + k) for k in range(3)]))
HS, n = ctx.bch(G, H)
DG, m = ctx.magnus_expand(ctx.op(-1, np.stack([random_operator(B, -1, 30 + k) for k in range(3)])), G)
print(n, m, HS.download().tobytes().hex(), DG.download().tobytes().hex())
"""


@pytest.mark.parametrize("wave", [0, 1, 3])
def test_series_gates(wave):
    assert run(SERIES, IMSRG_EMU_SPLIT=wave) == in_order(SERIES)


HF = """
H = E.Context(Basis.ho(2, 1)).op(1, synthetic_hamiltonian(Basis.ho(2, 1), 0))
D, e, n = H.hartree_fock()
print(e, n, np.asarray(D).tobytes().hex(), H.download().tobytes().hex())
"""


@pytest.mark.parametrize("wave", [0, 1, 3])
def test_hartree_fock_convergence(wave):
    assert run(HF, IMSRG_EMU_SPLIT=wave) == in_order(HF)
