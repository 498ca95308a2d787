"""The stage kernel compiled for cubic anisotropy with uniform exchange, against
the CPU oracle, with each neighbour of its rule: without exchange, with uniaxial
anisotropy and spin torque, per-cell cubic constant, and per-cell Ms (which takes
the general kernel); and as members of one batched launch."""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT, gpu_available, random_unit_field, rel_err

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import oracle as O  # noqa: E402

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

DELTA = (2e-9, 2.5e-9, 3e-9)


def physics(kind, shape):
    nx, ny, nz = shape
    kw = dict(Ms=8e5, alpha=0.3, A=1.3e-11, k_cub=-5e4, axis1=(1.0, 0.0, 0.0), axis2=(0.0, 1.0, 0.0))
    rng = np.random.default_rng(3)
    if kind == "no_exchange":
        del kw["A"]
    elif kind == "uniaxial_torque":
        kw.update(k_uni=3e5, P=0.7, xi=0.05, j=(1e12, 0.0, 0.0))
    elif kind == "per_cell_k":
        kw["k_cub"] = -5e4 * rng.uniform(0.5, 1.5, (nz, ny, nx))
    elif kind == "per_cell_ms":
        kw["Ms"] = 8e5 * (rng.random((nz, ny, nx)) > 0.2)
    return kw


KINDS = ["plain", "no_exchange", "uniaxial_torque", "per_cell_k", "per_cell_ms"]
# an even mesh, one with odd rows and a half-filled wave, and a single layer
SHAPES = [(32, 16, 4), (37, 9, 3), (70, 11, 1)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape", SHAPES)
def test_cubic_stage_vs_oracle(shape, kind):
    from micromagnum_amd.solver import Stepper
    kw = physics(kind, shape)
    M = random_unit_field(shape, 8) * np.asarray(kw["Ms"])
    st = Stepper(shape, DELTA, precision="fp64", method="rkf45", h0=2e-14, normalize_mode=1, **kw)
    st.set_m(M)
    dM, H = st.dmdt()
    sysO = O.System(shape, DELTA, N=st.N, **kw)
    dMo, Ho = sysO.dmdt(M)
    # some tens of roundings per cell, as the other dM/dt comparisons
    assert rel_err(H, Ho) < 1e-12 and rel_err(dM, dMo) < 1e-12
    E, Eo = st.energy(), sysO.energy(M)
    for k in ("E_aniso", "E_tot"):
        assert abs(E[k] - Eo[k]) <= 1e-12 * sum(abs(Eo[q]) for q in ("E_stray", "E_exch", "E_aniso", "E_ext")), k
    # FP32 of the same: 2^-24 times the same count of roundings
    st32 = Stepper(shape, DELTA, precision="fp32", method="rkf45", h0=2e-14, **kw)
    st32.set_m(M)
    dM32, H32 = st32.dmdt()
    assert rel_err(H32, Ho) < 1e-5 and rel_err(dM32, dMo) < 1e-5


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_cubic_members_of_a_batch(precision, monkeypatch):
    # every class side by side in one batch: the members step as they do alone
    from micromagnum_amd.solver import Ensemble, Stepper
    specs = [dict(shape=sh, delta=DELTA, method="rkf45", precision=precision, **physics(k, sh))
             for k in KINDS + ["plain"] for sh in SHAPES[:2]]
    specs[-1] = dict(specs[-1], k_uni=2e5)
    del specs[-1]["k_cub"], specs[-1]["axis2"]
    Ms = [random_unit_field(s["shape"], 20 + i) * np.asarray(s["Ms"]) for i, s in enumerate(specs)]
    monkeypatch.setenv("MM_BATCH_LAUNCH", "1")
    ens = Ensemble(specs)
    for i, M in enumerate(Ms):
        ens.set_m(i, M)
    ens.run(4)
    monkeypatch.setenv("MM_FFT_GENERIC", "1")  # the batch's z form (LDS) alone too
    for i, s in enumerate(specs):
        kw = {k: v for k, v in s.items() if k not in ("shape", "delta")}
        st = Stepper(s["shape"], s["delta"], N=ens.specs[i].N, **kw)
        st.set_m(Ms[i])
        st.run(4)
        tol = 1e-13 if precision == "fp64" else 1e-5
        assert rel_err(ens.get_m(i), st.get_m()) < tol, i
