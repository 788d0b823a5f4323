"""A HIP error that a call has reported does not come back from the next call (HIP keeps the last error of a thread,
and the checks after kernel launches read it)."""
import ctypes as C

import numpy as np
import pytest

import mlem_amd as M
from matrices import make

pytestmark = pytest.mark.gpu


def test_calls_after_a_refused_allocation():
    A = make("ragged", seed=3)
    AT = M.transpose(A)
    p = C.c_void_p()
    for _ in range(2):
        assert M.hip_lib().mlem_device_alloc(C.byref(p), 1 << 45) == 3  # out of memory
        with M.ResidentMatrix(A) as m:
            m.build_transpose()
            T = m.download_transpose()
        assert np.array_equal(T.rowptr, AT.rowptr) and np.array_equal(T.col, AT.col)
