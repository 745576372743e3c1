"""Launch schedules and variants are what the caller set, at every batch size, and none changes a
result: the sizes and MPDATA instances of small batches (levels dealt to workgroups) and of batches
that fill the device, the register-bounded MPDATA that the largest batches take by default among
them."""
import numpy as np
import pytest

from crm_hip import KERNELS, CrmHip, DeviceCase
from crm_inputs import add_convection, make_case
from crm_views import CrmDims
from test_gpu_chunks import repeated

pytestmark = pytest.mark.gpu

SIZED = ("init", "kurant", "pre", "sgs", "mom", "mpdata", "diffuse", "micro", "stats", "final")


def _run(hip, case, steps):
    dc = DeviceCase(case.copy(), "cuda:0")
    hip.run_device(dc, steps * case.dt)
    return dc.download()


def _same(a, b, n=None):
    for g in ("state", "rad", "out"):
        for k, v in getattr(a, g).items():
            assert np.array_equal(v[:n], getattr(b, g)[k][:n]), (g, k)


def _case(n, nx, nz, ny=1, dt=20.0):
    return add_convection(make_case(n, nx, nz, 4000.0, dt, ny=ny, randomize=True), seed=nx + nz)


# 7 and 16 waves, and 1024 (none of whose scalar sweeps is cut); an instance count that leaves a
# workgroup of every size partly empty
@pytest.mark.parametrize("shape", [(7, 64, 17, 1), (61, 16, 28, 1), (16, 8, 9, 8), (4097, 16, 9, 1)],
                         ids=lambda s: "x".join(str(v) for v in s))
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_sizes_set_are_the_sizes_launched(shape, prec):
    n, nx, nz, ny = shape
    case = _case(n, nx, nz, ny)
    small = n * nx * ny < 64 * 1024
    with CrmHip(0, prec) as hip:
        ref = _run(hip, case, 4)
        for k in SIZED:
            assert hip.launch_shape(case.dims(), k)[0] == (64 if small else hip.schedule()[k])
        for threads in (64, 128, 192, 256):
            hip.set_schedule({k: threads for k in KERNELS})
            for k in SIZED:
                assert hip.launch_shape(case.dims(), k)[0] == threads
            _same(ref, _run(hip, case, 4))


@pytest.mark.parametrize("shape", [(3, 64, 17, 1), (1025, 64, 9, 1), (1024, 8, 9, 8), (4100, 4, 9, 4), (520, 128, 8, 1)],
                         ids=lambda s: "x".join(str(v) for v in s))
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_mpdata_variants_are_the_ones_launched(shape, prec):
    n, nx, nz, ny = shape
    case = _case(n, nx, nz, ny)
    small = n * nx * ny < 64 * 1024
    with CrmHip(0, prec) as hip:
        ref = _run(hip, case, 3)
        for v, kind in enumerate((0, 1, 2, 3, 0, 2)):
            hip.set_variants({"mpdata": v})
            _, chunks, split, got = hip.launch_shape(case.dims(), "mpdata")
            assert got == kind and split == (small and v == 0) and (split or chunks == 1)
            _same(ref, _run(hip, case, 3))


def test_pieces_of_the_microphysics():
    """A full device takes two pieces per wave of columns (each adds an atomic maximum to the queued
    call), a smaller batch as many as give 8192 waves."""
    with CrmHip(0) as hip:
        for n, pieces in ((8192, 2), (4096, 2), (4095, 2), (2048, 4), (1024, 8), (64, 58)):
            assert hip.launch_shape(CrmDims(n, n, 60, 64, 1, 58, 16, 1, 1000.0, 5.0), "micro")[1] == pieces


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_default_mpdata_of_the_largest_batches(prec):
    """From 2048 waves of 64 columns on the registers are bounded: the bits of the small batch."""
    case = _case(2, 64, 11)
    big = repeated(case, 1024)
    with CrmHip(0, prec) as hip:
        assert hip.launch_shape(big.dims(), "mpdata")[3] == 2
        assert hip.launch_shape(case.dims(), "mpdata")[2] == 1
        _same(_run(hip, case, 4), _run(hip, big, 4), 2)


def test_autotuner_tries_what_the_batch_launches():
    """A small batch keeps the MPDATA whose levels are dealt, and the classes that the schedule does
    not size keep their defaults."""
    case = _case(16, 64, 28)
    with CrmHip(0) as hip, CrmHip(0) as ref:
        sched = hip.autotune(DeviceCase(case.copy(), "cuda:0"), 3 * case.dt)
        assert hip.variants()["mpdata"] == 0
        for k in ("setup", "setperturb", "precip_init", "press", "precip"):
            assert sched[k] == ref.schedule()[k]
        for k in SIZED:
            assert hip.launch_shape(case.dims(), k)[0] == sched[k]
        _same(_run(ref, case, 4), _run(hip, case, 4))
