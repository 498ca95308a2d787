"""Magnetisation read back through the pinned pieces: round trips at the edges of
the rule and of a piece, in both precisions, and from several threads at once."""
import threading

import numpy as np
import pytest

from conftest import gpu_available, random_unit_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]


def stepper(shape, precision, M):
    from micromagnum_amd.solver import Stepper
    st = Stepper(shape, (2e-9, 2e-9, 2e-9), precision=precision, Ms=8e5, alpha=0.5, A=1.3e-11, demag=False)
    st.set_m(M)
    return st


# 24 bytes a cell against 8 MiB; pieces of 2 MiB (524288 floats, 262144 doubles)
SHAPES = [(349525, 1, 1), (349526, 1, 1), (2 ** 19, 1, 1), (2 ** 19, 1, 2), (257, 255, 9), (1013, 701, 1)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_round_trip(shape, precision):
    M = random_unit_field(shape, 3) * 8e5
    st = stepper(shape, precision, M)
    want = M if precision == "fp64" else M.astype(np.float32).astype(np.float64)
    for _ in range(2):
        assert np.array_equal(st.get_m(), want)


def test_threads_side_by_side():
    shapes = [(257, 255, 9), (300, 200, 7), (1013, 701, 1)]
    Ms = [random_unit_field(s, i) * 8e5 for i, s in enumerate(shapes)]
    sts = [stepper(s, p, M) for s, M, p in zip(shapes, Ms, ("fp32", "fp64", "fp32"))]
    bad = []

    def read(i):
        want = Ms[i] if i == 1 else Ms[i].astype(np.float32).astype(np.float64)
        for _ in range(5):
            if not np.array_equal(sts[i].get_m(), want):
                bad.append(i)

    ts = [threading.Thread(target=read, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
