"""The y passes' narrow plans (540, 648, 900 and 1000 points on meshes that fill the
chip) against numpy's FFT in 64 bits, on either side of their rule, and in batches
against single steppers."""
import numpy as np
import pytest

from conftest import gpu_available, random_unit_field, rel_err
from test_gpu_compiled_lengths import numpy_field
from test_gpu_mixed_lengths import tensor

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]


# 2-D tiles of one column: 257 of them, 255 and 256 beside; 3-D tiles of two or four
@pytest.mark.parametrize("length", [540, 648, 900, 1000])
@pytest.mark.parametrize("nx,nz", [(256, 1), (250, 1), (240, 1), (45, 9), (64, 6), (20, 2)])
def test_narrow_lengths(nx, nz, length):
    from micromagnum_amd import magneto as mg
    from micromagnum_amd.device import empty, to_device
    shape = (nx, length // 2, nz)
    N = tensor(shape, length, 1)
    M = random_unit_field(shape, length) * 8e5
    ref = numpy_field(N, M)
    # a few roundings per pass: below 20 eps of the field's norm
    for precision, dtype, tol in (("fp64", np.float64, 1e-14), ("fp32", np.float32, 3e-6)):
        conv = mg.SymmetricMatrixVectorConvolution_FFT(N, *shape, precision=precision)
        assert conv.fft_size[1] == length
        H = empty(M.shape, dtype)
        conv.execute(to_device(M, dtype), H)
        assert rel_err(H.numpy(), ref) < tol, precision


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_narrow_members_of_a_batch(precision):
    from micromagnum_amd.solver import Ensemble, Stepper
    kw = dict(delta=(2e-9, 2.5e-9, 3e-9), method="rkf45", precision=precision, Ms=8e5, alpha=0.3, A=1.3e-11)
    shapes = [(256, 270, 1), (64, 324, 6), (40, 450, 2), (45, 30, 1)]
    specs = [dict(kw, shape=s) for s in shapes]
    ens = Ensemble(specs)
    Ms = [random_unit_field(s, i) * 8e5 for i, s in enumerate(shapes)]
    for i, M in enumerate(Ms):
        ens.set_m(i, M)
    ens.run(3)
    for i, s in enumerate(shapes):
        st = Stepper(s, N=ens.specs[i].N, **kw)
        st.set_m(Ms[i])
        st.run(3)
        assert np.array_equal(ens.get_m(i), st.get_m()), s
        st.close()
    ens.close()
