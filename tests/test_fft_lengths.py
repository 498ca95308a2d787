"""Transform lengths the library refuses, before anything is allocated (no GPU)."""
import ctypes

import numpy as np
import pytest

from micromagnum_amd import _lib


@pytest.mark.parametrize("n,message", [(3 ** 9, "passes"), (3 ** 16, "passes"), (3 ** 17, "passes"), (3 ** 19, "passes"),
                                       (2 * 3 ** 17, "passes"), (5 ** 13, "passes")])
def test_lengths_with_too_many_factors(n, message):
    # periodic along x, whose tensor has the mesh's own size; it is not read
    L = _lib.load()
    N, h = np.zeros(6), ctypes.c_void_p()
    rc = L.mm_conv_create(N.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), n, 1, 1, n, 1, 1, _lib.MM_FP64,
                          ctypes.byref(h))
    assert rc != _lib.MM_OK and not h.value
    assert message in L.mm_last_error().decode()
