"""Sedimentation in several sub-steps per substep where a column's levels are dealt to chunks (small
batches): the chunks of a workgroup meet between sub-steps, and 128-column instances, whose chunks
are workgroups that cannot meet, do all levels in one.  Odd and even counts (the field changes
buffers every sub-step), bitwise the sweep of a batch that fills the device."""
import numpy as np
import pytest

from crm_hip import CrmHip, DeviceCase
from crm_inputs import make_case
from test_gpu_chunks import repeated

pytestmark = pytest.mark.gpu


# columns, levels, substep [s], rain water [kg/kg] and the sub-steps it takes in the thinnest layer
@pytest.mark.parametrize("nx,ny,nz,dt,rain,count", [
    (128, 1, 58, 10.0, 2e-3, 2), (128, 1, 58, 20.0, 2e-3, 3), (128, 1, 58, 20.0, 2e-2, 5), (128, 1, 28, 20.0, 2e-2, 3),
    (64, 1, 58, 20.0, 2e-2, 5), (64, 1, 58, 10.0, 2e-3, 2), (16, 1, 40, 20.0, 0.1, 4), (8, 1, 58, 30.0, 2e-2, 7),
    (8, 8, 58, 20.0, 2e-3, 3), (4, 4, 58, 20.0, 2e-2, 5)], ids=lambda v: str(v))
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_sedimentation_substeps(nx, ny, nz, dt, rain, count, prec):
    case = make_case(2, nx, nz, 1000.0 if nz == 58 else 2000.0 if nz == 40 else 4000.0, dt, ny=ny, randomize=True)
    low = case.state["qp"][..., :nz // 2]
    low[...] = rain * np.random.default_rng(1).random(low.shape)
    times = -(-64 * 1024 // (2 * nx * ny))
    big = repeated(case, times)
    got = []
    with CrmHip(0, prec) as hip:
        assert hip.launch_shape(case.dims(), "precip")[1] > 1 and hip.launch_shape(big.dims(), "precip")[1] == 1
        for c in (case, big):
            dc = DeviceCase(c.copy(), "cuda:0")
            hip.run_device(dc, 3 * dt)
            assert (hip.stats().ncycle_max, hip.stats().nprec_max) == (1, count)
            got.append(dc.download())
    for group in ("state", "rad", "out"):
        for k, v in getattr(got[0], group).items():
            w = getattr(got[1], group)[k]
            assert np.array_equal(v, w[:2]) and np.array_equal(v, w[-2:]), (group, k)
