"""Host streams to and from the device: bit-identical round trips and the
hermitian mirror, for sizes packed on the host and on the device, batches,
sub-blocks that end inside a 32 x 32 tile, and streams long enough for the
copy ring (more than eight 4 MiB chunks)."""
import numpy as np
import pytest

from imsrg_mi355x import Basis, random_operator
from test_gpu_small_path import basis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("herm", [1, -1])
@pytest.mark.parametrize("emax,kp,kn,nb", [(1, 1, 1, 1), (2, 1, 3, 1), (3, 1, 6, 1), (3, 3, 1, 3), (5, 3, 6, 1), (7, 3, 6, 2)])
def test_operator_stream_round_trip(emax, kp, kn, nb, herm):
    from imsrg_mi355x import engine as E
    B = basis(emax, kp, kn)
    ctx = E.Context(B, nbatch=nb)
    v = np.stack([random_operator(B, herm, 3 + k) for k in range(nb)])
    A = ctx.op(herm, v)
    assert np.array_equal(A.download().reshape(nb, -1), v)
    # the mirror: the Frobenius norm counts both triangles and both one-body halves
    for k in range(nb):
        _, f, mats = B.full_from_vec(v[k], herm)
        want = np.sqrt((f * f).sum() + sum((m * m).sum() for m in mats))
        assert abs(np.atleast_1d(A.norm())[k] - want) <= 1e-13 * want


@pytest.mark.parametrize("emax,kp,kn,rank,dpar", [(2, 1, 1, 2, 2), (3, 1, 3, 4, 0), (7, 3, 3, 4, 0)])
def test_tensor_stream_round_trip(emax, kp, kn, rank, dpar):
    from imsrg_mi355x import engine as E
    B = basis(emax, kp, kn)
    T = E.Context(B).tensor(rank, dpar, 1)
    v = np.random.default_rng(emax).uniform(-1, 1, T.neq)
    assert np.array_equal(T.upload(v).download(), v)


def test_uploads_back_to_back():
    """an upload may return before the device has read its staging copy"""
    from imsrg_mi355x import engine as E
    B = Basis.ho(6, 3)
    ctx = E.Context(B)
    vs = [random_operator(B, 1, k) for k in range(4)]
    ops = [ctx.op(1, v) for v in vs]
    for o, v in zip(ops, vs):
        assert np.array_equal(o.download(), v)
