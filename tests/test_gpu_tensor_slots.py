"""The scalar-tensor series where a class's slot scan ends in an empty batch
(rank 4 at emax 3 and 4), against the m-scheme; the bound is
test_gpu_tensor_ranks'."""
import pytest

from test_gpu_tensor_ranks import test_series_against_m_scheme as series

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("emax,shells,rank,dpar", [(3, 3, 4, 0), (3, 1, 4, 2), (4, 1, 4, 0)])
def test_empty_batches(emax, shells, rank, dpar):
    series(emax, shells, rank, dpar)
