"""Every mixed-radix length with a compiled transform, along x, y and z, in
both precisions, against numpy's FFT in 64 bits; and one periodic axis of such
a length (a full line, no zero padding)."""
import numpy as np
import pytest

from conftest import gpu_available, random_unit_field, rel_err

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

Z = [6, 10, 12, 18, 20, 24, 30, 36, 40, 48, 50, 54, 60, 72, 80, 90, 96, 100, 108, 120]
XY = [144, 150, 160, 162, 180, 192, 200, 216, 240, 250, 270, 288, 300, 320, 324, 360, 384, 400, 432, 450, 480, 486,
      500, 540, 576, 600, 640, 648, 720, 750, 768, 800, 900, 960, 1000]


def numpy_field(N, M):
    nz, ny, nx = M.shape[1:]
    P = N.shape[:3]
    F = [np.fft.rfftn(M[c], s=P, axes=(0, 1, 2)) for c in range(3)]
    K = [np.fft.rfftn(N[..., e], axes=(0, 1, 2)) for e in range(6)]
    rows = [(0, 1, 2), (1, 3, 4), (2, 4, 5)]
    return np.stack([np.fft.irfftn(sum(K[e] * F[c] for c, e in enumerate(r)), s=P, axes=(0, 1, 2))[:nz, :ny, :nx]
                     for r in rows])


def check(shape, length, axis, pbc=(False, False, False)):
    from micromagnum_amd import magneto as mg
    from micromagnum_amd.device import empty, to_device
    nx, ny, nz = shape
    N = mg.GenerateDemagTensor(nx, ny, nz, 2e-9, 3e-9, 2.5e-9, *pbc, repeat=1)
    if not any(pbc):
        # the length itself, whatever the padding policy picks: more zeros
        ext = [N.shape[2], N.shape[1], N.shape[0]]
        ext[axis] = length
        big = np.zeros((ext[2], ext[1], ext[0], 6))
        idx = [np.arange(-(n - 1), n) for n in (nz, ny, nx)]
        big[np.ix_(*idx)] = N[np.ix_(*idx)]
        N = big
    M = random_unit_field(shape, length) * 8e5
    ref = numpy_field(N, M)
    for precision, dtype, tol in (("fp64", np.float64, 1e-14), ("fp32", np.float32, 3e-6)):
        conv = mg.SymmetricMatrixVectorConvolution_FFT(N, nx, ny, nz, precision=precision)
        assert conv.fft_size[axis] == length
        H = empty((3, nz, ny, nx), dtype)
        conv.execute(to_device(M, dtype), H)
        # a few roundings per pass: below 20 eps of the field's norm
        assert rel_err(H.numpy(), ref) < tol, (shape, precision)


@pytest.mark.parametrize("length", Z + XY)
def test_compiled_length(length):
    for axis in range(3 if length in Z else 2):
        shape = [3, 2, 2]
        shape[axis] = length // 2
        check(tuple(shape), length, axis)


@pytest.mark.parametrize("length", [12, 60, 150, 200])
def test_compiled_length_periodic(length):
    check((length, 3, 2), length, 0, (True, False, False))
    check((3, length, 2), length, 1, (False, True, False))
