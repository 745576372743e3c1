"""A call with mean-state acceleration queues all its substeps at once and lets the device stop at
the first that the host has to take over.  Bitwise the call whose host decides every substep
(CRM_GRAPHS_OFF): undisturbed, taken over at the first, a middle and the last substep, and with
heating strong enough for the 5 K test that ends the acceleration."""
import numpy as np
import pytest

from crm_hip import CrmHip, DeviceCase
from crm_inputs import add_convection, make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heating", [0.0, 0.02, 1.0])
@pytest.mark.parametrize("stop_at", [0, 1, 5, 10])
@pytest.mark.parametrize("shape", [(5, 32, 1, 28, "fp64"), (2, 8, 8, 33, "mixed")], ids=["32x28", "8x8x33_mixed"])
def test_accelerated_call_queued_whole(shape, stop_at, heating):
    n, nx, ny, nz, prec = shape
    case = make_case(n, nx, nz, 4000.0, 20.0, ny=ny, randomize=True)
    if heating:
        case = add_convection(case, seed=nz)
    case.rad["qrad"][...] = heating
    got = []
    for mode in (0, 2):
        with CrmHip(0, prec) as hip:
            hip.set_graphs(mode)
            hip.accel_init(True, 1.0, True)
            hip.debug_stop_call_at(stop_at if mode else 0)
            dc = DeviceCase(case.copy(), "cuda:0")
            counts = []
            for _ in range(2):  # the second call is heated by what the first has computed
                hip.run_device(dc, 400.0)
                st = hip.stats()
                counts.append((st.nstop, st.ncycle_max, st.accel_ceased))
            assert heating < 1.0 or counts[0][2]
            got.append((dc.download(), counts))
    assert got[0][1] == got[1][1]
    for group in ("state", "rad", "out"):
        for k, v in getattr(got[0][0], group).items():
            assert np.array_equal(v, getattr(got[1][0], group)[k], equal_nan=True), (group, k)
