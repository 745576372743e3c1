"""View structs from dicts of addresses: integers, null pointers and host arrays give the pointers
that CrmCase.views() makes of the same arrays."""
import ctypes as C

import numpy as np
import pytest

from crm_inputs import make_case
from crm_views import views_from_addresses


def _addresses(views):
    return [[C.cast(getattr(v, f), C.c_void_p).value for f, _ in v._fields_] for v in views]


@pytest.mark.parametrize("ncrms", [1, 3])
def test_addresses_arrays_and_nulls_mix(ncrms):
    case = make_case(ncrms, 8, 28, 4000.0, 20.0)
    groups = [dict(case.inp), dict(case.state), dict(case.rad), dict(case.out)]
    want = _addresses(case.views())
    as_int = [{k: None if v is None else v.ctypes.data for k, v in g.items()} for g in groups]
    mixed = [{k: (v if j % 2 else as_int[i][k]) for j, (k, v) in enumerate(g.items())} for i, g in enumerate(groups)]
    numpy_int = [{k: None if v is None else np.uint64(v) for k, v in g.items()} for g in as_int]
    for given in (groups, as_int, mixed, numpy_int):
        assert _addresses(views_from_addresses(*given)) == want
    no_rad = [as_int[0], as_int[1], {k: None for k in as_int[2]}, as_int[3]]
    assert _addresses(views_from_addresses(*no_rad))[2] == [None] * len(as_int[2])


def test_arrays_are_still_checked():
    case = make_case(2, 8, 28, 4000.0, 20.0)
    bad = dict(case.state, temperature=case.state["temperature"].astype(np.float32))
    with pytest.raises(AssertionError):
        views_from_addresses(case.inp, bad, case.rad, case.out)
