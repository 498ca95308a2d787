"""Members of an ensemble are single steppers bit for bit, also where the single
stepper runs its z lines in registers and the batched launch in LDS (6, 10, 12 and 16
points), and with mixed-radix lines along x and y."""
import numpy as np
import pytest

from conftest import gpu_available, random_unit_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

# (shape, tensor padding): the padding to a multiple of 2 gives 6- and 10-point z lines
MEMBERS = [((33, 18, 3), 1), ((40, 25, 5), 1), ((50, 27, 5), 2), ((45, 30, 6), 2), ((24, 20, 8), 2),
           ((60, 36, 2), 2), ((81, 50, 4), 2), ((54, 45, 1), 2)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["uniaxial", "percell"])
def test_members_are_single_steppers(kind, precision):
    from micromagnum_amd.solver import Ensemble, Stepper
    specs = []
    # FP32 lines of 16 points take registers on meshes with enough rows only
    members = MEMBERS + ([((200, 170, 8), 2)] if precision == "fp32" else [])
    for i, (shape, padding) in enumerate(members):
        kw = dict(shape=shape, delta=(2e-9, 2.5e-9, 3e-9), padding=padding, method="rkf45", precision=precision, Ms=8e5,
                  alpha=0.3, A=1.3e-11, k_uni=3e5, axis1=(0.6, 0.0, 0.8), h_ext=(1e4, 2e4, 0.0))
        if kind == "percell":
            kw["Ms"] = 8e5 * (1.0 + 0.25 * (np.arange(np.prod(shape)) % 3)).reshape(shape[::-1])
        specs.append(kw)
    ens = Ensemble(specs)
    Ms = [random_unit_field(s["shape"], i) * s["Ms"] for i, s in enumerate(specs)]
    for i, M in enumerate(Ms):
        ens.set_m(i, M)
    ens.run(5)
    for i, s in enumerate(specs):
        st = Stepper(s["shape"], N=ens.specs[i].N, **{k: v for k, v in s.items() if k not in ("shape", "padding")})
        st.set_m(Ms[i])
        st.run(5)
        assert np.array_equal(ens.get_m(i), st.get_m()), members[i]
        assert ens.stats(i) == st.stats(), members[i]
        st.close()
    ens.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape,length", [((400, 330, 5), 12), ((400, 330, 3), 8), ((120, 90, 6), 12)])
def test_register_lines_have_the_bits_of_the_others(shape, length, precision, monkeypatch):
    # on both sides of the workgroup sizes' rule (2^18 columns)
    from micromagnum_amd import magneto as mg
    from micromagnum_amd.device import empty, to_device
    N = mg.GenerateDemagTensor(*shape, 2e-9, 2.5e-9, 3e-9, device="gpu")
    dt = np.float64 if precision == "fp64" else np.float32
    M = to_device(random_unit_field(shape, 3) * 8e5, dt)
    out = []
    for generic in ("0", "1"):
        monkeypatch.setenv("MM_FFT_GENERIC", generic)
        conv = mg.SymmetricMatrixVectorConvolution_FFT(N, *shape, precision=precision)
        assert conv.fft_size[2] == length
        H = empty(M.shape, dt)
        conv.execute(M, H)
        out.append(H.numpy())
    assert np.array_equal(out[0], out[1])
