"""Threads of the stage kernel on meshes of long rows that fill the chip: the count
that keeps 1536 threads on a CU (FP32), which the kernels' registers must leave room
for -- two workgroups of 768 with 1024-cell rows, three of 512 with 512-cell rows."""
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

STT = dict(P=0.7, xi=0.05, j=(1e12, 0.0, 0.0))
CUBIC = dict(k_cub=-5e3, axis1=(1.0, 0.0, 0.0), axis2=(0.0, 1.0, 0.0))


@pytest.mark.parametrize("shape,physics,threads", [((1024, 512, 2), STT, 768), ((1024, 512, 2), CUBIC, 768),
                                                   ((1024, 512, 2), {}, 768), ((512, 256, 16), STT, 512),
                                                   ((512, 256, 16), CUBIC, 512), ((512, 256, 16), {}, 512)])
def test_threads_on_long_rows(shape, physics, threads):
    from micromagnum_amd.solver import Stepper
    st = Stepper(shape, (2e-9, 2e-9, 2e-9), precision="fp32", Ms=8e5, alpha=0.1, A=1.3e-11, tensor="gpu", **physics)
    assert st.launch_shape()["stage_threads"] == threads
    st.close()
