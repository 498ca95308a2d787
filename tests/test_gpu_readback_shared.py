"""One stepper whose magnetisation several threads read at the same time: every
reader gets the state, whole (ctypes releases the interpreter lock during a read)."""
import threading

import numpy as np
import pytest

from conftest import gpu_available, random_unit_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(300, 200, 7), (1013, 701, 2)])
def test_readers_of_one_stepper(shape, precision):
    from micromagnum_amd.solver import Stepper
    M = random_unit_field(shape, 5) * 8e5
    st = Stepper(shape, (2e-9, 2e-9, 2e-9), precision=precision, Ms=8e5, alpha=0.5, A=1.3e-11, demag=False)
    st.set_m(M)
    want = M if precision == "fp64" else M.astype(np.float32).astype(np.float64)
    start, bad = threading.Barrier(3), []

    def read(i):
        start.wait(60)
        for _ in range(6):
            if not np.array_equal(st.get_m(), want):
                bad.append(i)

    ts = [threading.Thread(target=read, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
