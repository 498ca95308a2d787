"""The z pass in registers (short z lines) against numpy's FFT in 64 bits and
against the LDS form, at the edges of its rule: every length it takes, full and
part-filled lines, rows that end inside a wave, and lines it must leave alone."""
import numpy as np
import pytest

from conftest import gpu_available, random_unit_field, rel_err
from test_gpu_compiled_lengths import numpy_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]


def field(shape, length, precision, pbc=(False, False, False)):
    """H of a random field on the GPU and its 64-bit value; the tensor is
    embedded so that z lines have `length` points"""
    from micromagnum_amd import magneto as mg
    from micromagnum_amd.device import empty, to_device
    nx, ny, nz = shape
    N = mg.GenerateDemagTensor(nx, ny, nz, 2e-9, 3e-9, 2.5e-9, *pbc, repeat=1)
    if not any(pbc):
        big = np.zeros((length,) + N.shape[1:])
        k = np.arange(-(nz - 1), nz)
        big[k] = N[k]
        N = big
    M = random_unit_field(shape, length) * 8e5
    dt = np.float64 if precision == "fp64" else np.float32
    conv = mg.SymmetricMatrixVectorConvolution_FFT(N, nx, ny, nz, precision=precision)
    assert conv.fft_size[2] == length
    H = empty((3, nz, ny, nx), dt)
    conv.execute(to_device(M, dt), H)
    return H.numpy(), numpy_field(N, M)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-14), ("fp32", 3e-6)])
@pytest.mark.parametrize("shape,length", [
    ((16, 8, 2), 4), ((33, 7, 2), 6), ((5, 3, 3), 6), ((20, 9, 3), 8), ((31, 6, 4), 8), ((20, 9, 4), 10),
    ((20, 9, 5), 10), ((12, 40, 5), 12), ((17, 5, 6), 12),
    ((150, 128, 7), 16), ((200, 130, 8), 16),  # 16 points: enough rows for the register form in FP32
    ((20, 9, 8), 16), ((9, 6, 9), 18),         # and lines that stay in LDS
])
def test_short_z_lines(shape, length, precision, tol, monkeypatch):
    # a few roundings per pass: below 20 eps of the field's norm for both forms
    H, ref = field(shape, length, precision)
    assert rel_err(H, ref) < tol
    monkeypatch.setenv("MM_FFT_GENERIC", "1")
    L, _ = field(shape, length, precision)
    assert rel_err(L, ref) < tol and rel_err(H, L.astype(np.float64)) < tol


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-14), ("fp32", 3e-6)])
@pytest.mark.parametrize("nz", [4, 8, 12])
def test_periodic_z_lines_stay_whole(nz, precision, tol):
    # a periodic axis has no zero half: its lines must not take the form that reads half
    H, ref = field((10, 6, nz), nz, precision, (False, False, True))
    assert rel_err(H, ref) < tol


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("layers", [(2, 3, 4), (2, 5, 4, 9), (5, 12)])
def test_batch_of_short_z_lines(layers, precision, monkeypatch):
    # register and LDS lines in one batch: every member as it steps alone
    # (in the forms the batch takes: LDS beyond 8 points), bit for bit
    from micromagnum_amd.solver import Ensemble, Stepper
    kw = dict(delta=(2e-9, 2.5e-9, 3e-9), method="rkf45", precision=precision, Ms=8e5, alpha=0.5, A=1.3e-11)
    specs = [dict(kw, shape=(33 + 7 * i, 18 + i, nz)) for i, nz in enumerate(layers)]
    Ms = [random_unit_field(s["shape"], i) * 8e5 for i, s in enumerate(specs)]
    monkeypatch.setenv("MM_BATCH_LAUNCH", "1")
    ens = Ensemble(specs)
    for i, M in enumerate(Ms):
        ens.set_m(i, M)
    ens.run(5)
    for i, s in enumerate(specs):
        monkeypatch.setenv("MM_FFT_GENERIC", "1" if layers[i] > 4 else "0")
        st = Stepper(s["shape"], N=ens.specs[i].N, **{k: v for k, v in s.items() if k != "shape"})
        st.set_m(Ms[i])
        st.run(5)
        assert np.array_equal(ens.get_m(i), st.get_m()), i
