"""Exchange with per-cell Ms and A inside the stage kernel: a uniform state has no
exchange field and no exchange energy, not even the rounding of M / Ms, and in FP32
the error is that of the quotients of the neighbours a cell has.  Cells thinner than
wide, so that a direction without a neighbour has the largest weight."""
import numpy as np
import pytest

import oracle as O
from conftest import gpu_available, random_unit_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

MU0 = 4e-7 * np.pi


def material(shape, varied):
    """a disk in the mesh's plane; with `varied`, Ms differs from cell to cell"""
    nx, ny, nz = shape
    x, y = (np.arange(nx) + 0.5) / nx * 2 - 1, (np.arange(ny) + 0.5) / ny * 2 - 1
    on = np.broadcast_to(x[None, :] ** 2 + y[:, None] ** 2 < 1.0, (nz, ny, nx)).astype(np.float64)
    Ms = 8e5 * on
    if varied:
        Ms = Ms * np.random.default_rng(2).uniform(0.5, 1.5, on.shape)
    return Ms, 1.3e-11 * on


def stepper(shape, delta, precision, Ms, A, pbc=(False,) * 3):
    from micromagnum_amd.solver import Stepper
    return Stepper(shape, delta, precision=precision, method="rkf45", Ms=Ms, alpha=0.1, A=A, demag=False, pbc=pbc)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("shape,delta,pbc", [
    ((33, 20, 1), (5e-9, 5e-9, 5e-10), (False, False, False)),
    ((64, 9, 3), (4e-9, 4e-9, 1e-9), (False, False, False)),
    ((16, 16, 2), (2e-9, 3e-9, 1e-9), (True, False, False)),
])
def test_uniform_state_has_no_exchange(shape, delta, pbc, precision):
    Ms, A = material(shape, False)
    for d in ((0.6, -0.64, 0.48), (1.0 / 3.0, 2.0 / 3.0, -2.0 / 3.0), (0.0, 0.0, 1.0)):
        st = stepper(shape, delta, precision, Ms, A, pbc)
        st.set_m(np.array(d).reshape(3, 1, 1, 1) * Ms)
        dM, H = st.dmdt()
        assert np.all(H == 0.0) and np.all(dM == 0.0)
        assert st.energy()["E_exch"] == 0.0
        st.close()


@pytest.mark.parametrize("varied", [False, True])
@pytest.mark.parametrize("shape,delta", [((40, 40, 1), (4e-9, 4e-9, 1e-9)), ((40, 40, 1), (5e-9, 5e-9, 5e-10)),
                                         ((40, 33, 3), (3e-9, 3e-9, 4e-9))])
def test_fp32_error_is_that_of_the_quotients(shape, delta, varied):
    Ms, A = material(shape, varied)
    Ms32, A32 = (v.astype(np.float32).astype(np.float64) for v in (Ms, A))
    M = (random_unit_field(shape, 4) * Ms32).astype(np.float32).astype(np.float64)
    st = stepper(shape, delta, "fp32", Ms32, A32)
    st.set_m(M)
    _, H = st.dmdt()
    ref, _ = O.exchange(delta, Ms32, A32, M)
    # each neighbour's term (m_j - m_i) w: two quotients of at most 1, rounded to 2^-25
    # each, and the term itself (at most 2 w) with its weight, difference and sum
    # rounded by 2^-24 each; the factor 2 A / (mu0 Ms) with four roundings
    w = sum(2.0 / d ** 2 for d, n in zip(delta, shape) if n > 1)
    f = 2.0 * A32.max() / (MU0 * Ms32[Ms32 > 0].min())
    bound = f * w * (2 * 2.0 ** -25 + 2 * 8 * 2.0 ** -24) + 4 * 2.0 ** -24 * np.abs(ref).max()
    assert np.abs(H - ref).max() < bound
    # on a smooth state only the quotients count
    X = (np.arange(shape[0]) - 0.5 * shape[0])[None, None, :] + 0.0 * Ms
    Y = (np.arange(shape[1]) - 0.5 * shape[1])[None, :, None] + 0.0 * Ms
    v = np.stack([-Y, X, 40.0 + 0.0 * Ms])
    M = (v / np.sqrt((v ** 2).sum(0)) * Ms32).astype(np.float32).astype(np.float64)
    st.set_m(M)
    _, H = st.dmdt()
    ref, _ = O.exchange(delta, Ms32, A32, M)
    # neighbours differ by at most 0.05 here: the terms' own roundings are that much smaller
    bound = f * w * (2 * 2.0 ** -25 + 0.05 * 8 * 2.0 ** -24) + 4 * 2.0 ** -24 * np.abs(ref).max()
    assert np.abs(H - ref).max() < bound
