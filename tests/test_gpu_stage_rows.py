"""The stage kernel's epilogue walks rows over groups of whole waves: row
lengths around the wave size, odd row counts, single-layer and single-row
meshes, with uniform and per-cell material, two RKF45 steps against the
oracle (FP64, FP64 norm)."""
import numpy as np
import pytest

import oracle as O
from conftest import gpu_available, random_unit_field

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape", [(63, 5, 3), (64, 3, 2), (65, 7, 1), (130, 2, 2), (40, 9, 1), (1, 5, 4), (300, 1, 3)])
def test_stage_rows_vs_oracle(shape, masked):
    from micromagnum_amd.solver import Stepper
    nx, ny, nz = shape
    on = np.ones((nz, ny, nx))
    if masked:
        on[(np.arange(on.size) % 5 == 2).reshape(on.shape)] = 0.0
        on *= 1.0 + 0.25 * (np.arange(on.size) % 3).reshape(on.shape)
    kw = dict(Ms=8e5 * on, alpha=0.1, A=1.3e-11 * on, h_ext=(1e4, 2e4, 0.0))
    M = random_unit_field(shape, 17) * kw["Ms"]
    delta = (3e-9, 2e-9, 4e-9)
    st = Stepper(shape, delta, precision="fp64", method="rkf45", normalize_mode=1, **kw)
    st.set_m(M)
    st.run(2)
    sysO = O.System(shape, delta, N=st.N, normalize_mode=1, **kw)
    Mo, so = sysO.run(M, method="rkf45", steps=2)
    s = st.stats()
    assert s["attempts"] == so["attempts"] and s["rejections"] == so["rejections"]
    # two steps: rounding (1e-15 of M) through the step control's 1e3
    assert np.abs(st.get_m() - Mo).max() / 1.2e6 < 1e-11
    st.close()
