"""Accelerated calls queue their substeps without the host's decision, a few ahead of the device:
how many ran from the queue, where the device stopped it (the test hook, the 5 K test that ends the
acceleration in a middle substep and in the last one, a substep that needs subcycles), and that few
were launched behind the stop.  Every call bitwise the one whose host decides every substep."""
import numpy as np
import pytest

from crm_hip import CrmHip, DeviceCase
from crm_inputs import add_convection, make_case

pytestmark = pytest.mark.gpu

AHEAD = 4  # QUEUE_AHEAD of the library


def _call(case, prec, mode, dt_gl, stop_at=0):
    with CrmHip(0, prec) as hip:
        hip.set_graphs(mode)
        hip.accel_init(True, 1.0, True)
        hip.debug_stop_call_at(stop_at)
        dc = DeviceCase(case.copy(), "cuda:0")
        hip.run_device(dc, dt_gl)
        st = hip.stats()
        return dc.download(), (st.nstop, st.ncycle_max, st.accel_ceased), hip.queue_counts()


def _same(a, b):
    for g in ("state", "rad", "out"):
        for k, v in getattr(a, g).items():
            assert np.array_equal(v, getattr(b, g)[k]), (g, k)


SHAPES = [(5, 32, 1, 28, "fp64"), (2, 8, 8, 33, "mixed")]
IDS = ["32x28", "8x8x33_mixed"]


@pytest.mark.parametrize("stop_at", [0, 1, 2, 7, 20])
@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_where_the_queue_stops(shape, stop_at):
    n, nx, ny, nz, prec = shape
    case = make_case(n, nx, nz, 4000.0, 20.0, ny=ny, randomize=True)
    want, steps, counts = _call(case, prec, 0, 800.0)
    assert steps == (20, 1, 0) and counts == (0, 0)
    got, steps, (launched, ran) = _call(case, prec, 2, 800.0, stop_at)
    assert steps == (20, 1, 0)
    assert ran == (stop_at - 1 if stop_at else 20)
    # the stopped substep, and those launched before its decision was known
    assert launched <= min(20, ran + 1 + AHEAD)
    _same(want, got)


# substeps the call has without the 5 K flag, heating rate of the four lowest levels [K/s], and the
# substep in which a level's mean first changes by more than 5 K: a middle one; the first; the last
# one, whose flag only the host's look behind the queue finds
@pytest.mark.parametrize("shape,nstop,heating,step", [
    (SHAPES[0], 10, 0.2495, 8), ((2, 8, 8, 33, "fp64"), 10, 0.2495, 7), (SHAPES[1], 10, 1.0, 1), (SHAPES[0], 1, 1.0, 1),
    (SHAPES[1], 1, 1.0, 1)], ids=["middle", "middle_3d", "first_mixed", "last", "last_mixed"])
def test_five_kelvin_in_a_queued_substep(shape, nstop, heating, step):
    n, nx, ny, nz, prec = shape
    case = make_case(n, nx, nz, 4000.0, 20.0, ny=ny, randomize=True)
    case.rad["qrad"][..., :4] = heating
    want, steps, _ = _call(case, prec, 0, 40.0 * nstop)
    assert (steps[0], steps[2]) == (nstop + nstop - step + 1, 1)
    got, got_steps, (launched, ran) = _call(case, prec, 2, 40.0 * nstop)
    assert got_steps == steps and ran == step
    assert launched <= min(nstop, step + 1 + AHEAD)
    _same(want, got)


@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_subcycles_in_a_queued_call(shape):
    n, nx, ny, nz, prec = shape
    case = add_convection(make_case(n, nx, nz, 4000.0, 20.0, ny=ny, randomize=True), seed=nz)
    case.state["w_wind"][...] *= 3.0
    want, steps, _ = _call(case, prec, 0, 800.0)
    assert steps[1] >= 2
    got, got_steps, (launched, ran) = _call(case, prec, 2, 800.0)
    assert got_steps == steps and ran < 20 and launched <= min(20, ran + 1 + AHEAD)
    _same(want, got)
