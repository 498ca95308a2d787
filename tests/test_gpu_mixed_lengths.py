"""Mixed-radix lines where the plain convolution of a 3-D mesh does not reach: the y
pass of single-layer meshes and the x transforms of the stage kernel, for every
compiled length; and ensembles whose members include a length without a compiled
transform, which takes that pass of every member to the kernels that run the plans in
a loop."""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT, gpu_available, random_unit_field, rel_err
from test_gpu_compiled_lengths import XY, Z, numpy_field

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import oracle as O  # noqa: E402

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

DELTA = (2e-9, 3e-9, 2.5e-9)


def tensor(shape, length, axis):
    """the mesh's tensor in a grid with `length` points along an axis"""
    from micromagnum_amd import magneto as mg
    N = mg.GenerateDemagTensor(*shape, *DELTA)
    ext = [N.shape[2], N.shape[1], N.shape[0]]
    ext[axis] = length
    big = np.zeros((ext[2], ext[1], ext[0], 6))
    idx = [np.arange(-(n - 1), n) for n in shape[::-1]]
    big[np.ix_(*idx)] = N[np.ix_(*idx)]
    return big


# a few roundings per pass: below 20 eps of the field's norm
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-14), ("fp32", 3e-6)])
@pytest.mark.parametrize("length", Z + XY)
def test_single_layer_and_stage(length, precision, tol):
    from micromagnum_amd import magneto as mg
    from micromagnum_amd.device import empty, to_device
    from micromagnum_amd.solver import Stepper
    dt = np.float64 if precision == "fp64" else np.float32
    shape = (20, length // 2, 1)
    N = tensor(shape, length, 1)
    M = random_unit_field(shape, length) * 8e5
    conv = mg.SymmetricMatrixVectorConvolution_FFT(N, *shape, precision=precision)
    assert conv.fft_size[1] == length
    H = empty(M.shape, dt)
    conv.execute(to_device(M, dt), H)
    assert rel_err(H.numpy(), numpy_field(N, M)) < tol
    for shape in ((length // 2, 3, 1), (length // 2, 2, 3)):
        N = tensor(shape, length, 0)
        M = random_unit_field(shape, length) * 8e5
        st = Stepper(shape, DELTA, N=N, precision=precision, Ms=8e5, alpha=0.1)
        st.set_m(M)
        assert rel_err(st.dmdt()[1], numpy_field(N, M)) < tol
        st.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("odd", [(405, 4, 1), (4, 405, 1), (4, 405, 2), (5, 4, 72), (1, 7, 2), (9, 1, 3)])
def test_batch_with_a_length_outside_the_table(odd, precision):
    # 810 and 144 (as a z line) points, and lines of one point
    from micromagnum_amd.solver import Ensemble, Stepper
    kw = dict(delta=DELTA, method="rkf45", precision=precision, Ms=8e5, alpha=0.3, A=1.3e-11, h0=2e-14, normalize_mode=1)
    specs = [dict(kw, shape=s) for s in (odd, (45, 30, 3), (81, 27, 1), (48, 20, 6), (135, 6, 12), (32, 16, 2))]
    ens = Ensemble(specs)
    Ms = [random_unit_field(s["shape"], 7 + i) * 8e5 for i, s in enumerate(specs)]
    for i, M in enumerate(Ms):
        ens.set_m(i, M)
    ens.run(3)
    for i, s in enumerate(specs):
        rest = {k: v for k, v in s.items() if k not in ("shape", "delta")}
        st = Stepper(s["shape"], DELTA, N=ens.specs[i].N, **rest)
        st.set_m(Ms[i])
        st.run(3)
        assert np.array_equal(ens.get_m(i), st.get_m()), s["shape"]
        st.close()
        if precision == "fp64":
            sysO = O.System(s["shape"], DELTA, N=ens.specs[i].N, Ms=8e5, alpha=0.3, A=1.3e-11, normalize_mode=1)
            Mo, so = sysO.run(Ms[i], method="rkf45", steps=3, h0=2e-14)
            assert ens.stats(i)["attempts"] == so["attempts"]
            # as the other ensemble members against the oracle
            assert np.abs(ens.get_m(i) - Mo).max() / 8e5 < 1e-10
    ens.close()
