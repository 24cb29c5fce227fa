"""Operator calls at the edges of what they accept: empty rows, empty contractions, and shapes on either side of a kernel's limit."""
import ctypes as C

import numpy as np
import pytest

from spy_amd import _lib as H
from tests import oracle_lib as O

B = C.byref


@pytest.mark.parametrize("exact", [0, 1])
@pytest.mark.parametrize("ne", [[0, 3], [0, 1], [0, 2, 2, 5]])
def test_norm_rms_of_empty_rows_launches_nothing(exact, ne):
    """NormRMS of rows without elements is accepted and does nothing, in either summation order: it returns before any device call, so the pointers
    here are never used (a launch would fail where there is no device and read before the rows where there is one)."""
    L = H.load()
    prev = L.spy_hip_set_exact_order(exact)
    try:
        assert L.spy_hip_op_norm_rms(None, B(H.tensor(4096, H.F32, ne)), B(H.tensor(8192, H.F32, ne)), 1e-5) == 0
        assert L.spy_hip_op_norm_rms(None, B(H.tensor(4096, H.F32, ne)), B(H.tensor(8192, H.F32, [0, 7])), 1e-5) == H.EINVAL
    finally:
        L.spy_hip_set_exact_order(prev)
