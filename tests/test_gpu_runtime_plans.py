"""MM_FFT_GENERIC=1 takes every pass, of single steppers and of batches, to the
kernels that run the transforms' passes in a loop, with their L/8 threads per line,
and gives the bits of the compiled transforms."""
import numpy as np
import pytest

from conftest import gpu_available, random_unit_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

KW = dict(delta=(2e-9, 2.5e-9, 3e-9), method="rkf45", Ms=8e5, alpha=0.3, A=1.3e-11)
# x lines of 324, 64, 90, 12 and 180 points; y and z lines mixed and powers of two
SHAPES = [(162, 9, 3), (32, 27, 5), (45, 32, 12), (6, 40, 1), (90, 81, 1)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_runtime_plans_run_and_agree(precision, monkeypatch):
    from micromagnum_amd.solver import Ensemble, Stepper
    specs = [dict(KW, shape=s, precision=precision) for s in SHAPES]
    Ms = [random_unit_field(s, i) * 8e5 for i, s in enumerate(SHAPES)]

    def single(i, N):
        st = Stepper(SHAPES[i], N=N, precision=precision, **KW)
        st.set_m(Ms[i])
        st.run(4)
        return st.get_m(), st.launch_shape()

    def batch():
        ens = Ensemble(specs)
        for i, M in enumerate(Ms):
            ens.set_m(i, M)
        ens.run(4)
        return [ens.get_m(i) for i in range(len(specs))], [s.N for s in ens.specs]

    want, tensors = batch()
    monkeypatch.setenv("MM_FFT_GENERIC", "1")
    got, _ = batch()
    for i, (nx, _, _) in enumerate(SHAPES):
        M, shape = single(i, tensors[i])
        points = 2 * nx
        assert shape["lpw_x"] == 256 // max(1, (points + 7) // 8)
        assert np.array_equal(M, want[i]) and np.array_equal(got[i], want[i]), SHAPES[i]
