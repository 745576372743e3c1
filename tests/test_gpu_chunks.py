"""Sweeps whose levels are dealt to several workgroups (small batches) give the bits of the sweep
over all levels (batches that fill the device): the same instances alone and repeated until the
batch is large enough that no scalar sweep is cut.  Copies change no batch-global maximum, so the
subcycle and sedimentation counts agree.  Shapes where a chunk can go wrong: the fewest levels, a
count no chunk divides, the compiled-in counts, the most; every lane geometry, and an instance
count that leaves a wave partly empty."""
import numpy as np
import pytest

import oracle_lib
from crm_hip import CrmHip, DeviceCase
from crm_inputs import add_convection, make_case
from parity import convective_case, relerr

pytestmark = pytest.mark.gpu

# ncrms, nx, ny, nz, dx, dt, substeps, precision
SHAPES = [(3, 64, 1, 8, 4000.0, 20.0, 4, "fp64"), (3, 32, 1, 28, 4000.0, 20.0, 6, "fp64"),
          (2, 64, 1, 58, 1000.0, 5.0, 6, "fp64"), (5, 16, 1, 33, 2000.0, 10.0, 4, "fp64"),
          (9, 8, 1, 11, 4000.0, 20.0, 4, "fp64"), (3, 128, 1, 29, 2000.0, 10.0, 4, "fp64"),
          (3, 8, 8, 28, 4000.0, 20.0, 4, "fp64"), (5, 4, 4, 64, 1000.0, 5.0, 4, "fp64"),
          (3, 64, 1, 28, 4000.0, 20.0, 4, "mixed"), (3, 128, 1, 58, 1000.0, 5.0, 3, "mixed"),
          (5, 16, 1, 9, 4000.0, 20.0, 4, "mixed"), (2, 8, 8, 41, 2000.0, 10.0, 3, "mixed")]


def repeated(case, times):
    """The instances of case, `times` copies of all of them."""
    big = make_case(case.ncrms * times, case.nx, case.nz, case.dx, case.dt, ny=case.ny, nx_rad=case.nx_rad,
                    ny_rad=case.ny_rad)
    for group in ("inp", "state", "rad", "out"):
        for k, v in getattr(case, group).items():
            getattr(big, group)[k][...] = np.concatenate([v] * times, axis=0)
    return big


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(str(v) for v in s))
def test_chunked_levels_give_the_same_bits(shape):
    n, nx, ny, nz, dx, dt, steps, prec = shape
    case = add_convection(make_case(n, nx, nz, dx, dt, ny=ny, randomize=True, nx_rad=nx // 2, ny_rad=ny), seed=nz)
    times = -(-64 * 1024 // (nx * ny * n))
    big = repeated(case, times)
    assert big.ncrms * nx * ny >= 64 * 1024
    got = {}
    for name, c in (("small", case), ("large", big)):
        dc = DeviceCase(c.copy(), "cuda:0")
        with CrmHip(0, prec) as hip:
            hip.run_device(dc, steps * dt)
            counts = (hip.stats().ncycle_max, hip.stats().nprec_max)
        got[name] = (dc.download(), counts)
    assert got["small"][1] == got["large"][1]
    for group in ("state", "rad", "out"):
        for k, v in getattr(got["small"][0], group).items():
            w = getattr(got["large"][0], group)[k]
            for first in (0, (times - 1) * n):  # the first and the last copy
                assert np.array_equal(v, w[first:first + n]), (group, k, first)


def test_sedimentation_substeps_of_a_chunked_column():
    """Several precipitation sub-steps per substep (heavy rain in thin layers under a long step):
    the chunks of a column exchange each sub-step's field."""
    case = add_convection(make_case(2, 32, 28, 4000.0, 20.0, randomize=True), seed=5)
    case.state["qp"][...] *= 4.0
    big = repeated(case, 1024)
    res = []
    for c in (case, big):
        dc = DeviceCase(c.copy(), "cuda:0")
        with CrmHip(0) as hip:
            hip.run_device(dc, 60.0)
            assert hip.stats().nprec_max >= 2
        res.append(dc.download())
    for group in ("state", "rad", "out"):
        for k, v in getattr(res[0], group).items():
            assert np.array_equal(v, getattr(res[1], group)[k][:2]), (group, k)


# The pressure solve's tiles of 16 levels (one level over and under a tile, the fewest, the most), its
# lane and column geometries, and instance counts that leave a workgroup partly empty.
@pytest.mark.parametrize("nx,nz,n", [(8, 8, 9), (8, 17, 7), (16, 16, 5), (16, 31, 3), (32, 33, 3), (32, 49, 1),
                                     (64, 8, 2), (64, 15, 1), (64, 48, 3), (64, 64, 2), (128, 9, 1), (128, 64, 2)])
def test_pressure_solve_at_tile_edges(nx, nz, n):
    """The first substep up to and with the pressure solve against the C restatement, within the
    parity bar of one substep (1e-10 of each field's largest value): the transform's sums of up to
    128 products and the sweep of up to 64 levels round at 1e-16 each.  Every variant gives the
    same bits."""
    dt = 20.0 * 28 / max(nz, 28)
    case = convective_case(n, nx=nx, nz=nz, dx=2000.0, dt=dt, seed=nx + nz)
    o = oracle_lib.oracle()
    assert o.run(case.copy(), dt, 13) == 0
    size = n * (nz + 1) * nx
    fields = ("u", "w", "dudt_na", "dwdt_na", "dudt_nc", "dwdt_nc")
    got = {}
    for variant in range(5 if nx == 64 else 1):
        with CrmHip(0) as hip:
            hip.set_variants({"press": variant})
            assert hip.debug_run(case.copy(), dt, 13) == 0
            got[variant] = {f: hip.debug_get(f, size).copy() for f in fields}
        for f in fields:
            assert np.array_equal(got[variant][f], got[0][f]), (variant, f)
    for f in fields:
        assert relerr(got[0][f], o.field(f, size)) <= 1e-10, f
