"""The scalar-tensor series over tensor ranks, against the m-scheme: where the
recoupling and Pandya kernels change form.  The smallest basis (work items of
one orbit quadruple), a parity-changing rank whose classes leave remainders in
the items, and a rank with more than 128 (J1, J2) outputs per quadruple.

Tolerance 1e-6 of the norm: the entries of the ph products below
float32(1e-6) are dropped, as TS_commutators.f90:1562, 1714 does, and the
m-scheme keeps them; everything else agrees to rounding.
"""
import importlib.util
import pathlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

_spec = importlib.util.spec_from_file_location("perf_cases", pathlib.Path(__file__).parents[1] / "perf" / "cases.py")
cases = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(cases)


@pytest.mark.parametrize("emax,shells,rank,dpar", [(1, 1, 2, 2), (3, 3, 6, 2), (4, 1, 32, 0)])
def test_series_against_m_scheme(emax, shells, rank, dpar):
    case = dict(name="t", op="tensor", emax=emax, kp=shells, kn=shells, rank=rank, dpar=dpar)
    got = cases.run(cases.prepare(case, 3))
    torch.cuda.synchronize()
    want = cases.exact(case, 3)["t"].numpy()
    t = np.asarray(got["t"].cpu() if torch.is_tensor(got["t"]) else got["t"])
    assert t.shape == want.shape
    assert np.linalg.norm(t - want) <= 1e-6 * np.linalg.norm(want)
