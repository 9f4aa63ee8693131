"""Step Jacobians of records that hold NaN, infinities or values out of any model's range: the rows of the sweep
through the whole step, NaN where it has them, though a row of an ordinary record is swept through a part."""
import ctypes

import numpy as np
import pytest

from test_group_host import LIB, N, inputs, params, run


def jacobians(flat, ovr, recs, ctl):
    lib = ctypes.CDLL(LIB)
    i, p = ctypes.c_int, ctypes.c_void_p
    lib.group_jacobian_run.argtypes = [i, p, i, p, p, i, p, p]
    out = [np.zeros((21, 24, N)) for _ in range(2)]
    for full in (0, 1):
        assert lib.group_jacobian_run(full, flat.ctypes.data, flat.size, ovr.ctypes.data, recs.ctypes.data, N,
                                      ctl.ctypes.data, out[full].ctypes.data) == 0
    return out


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 1e40, -1e200])
@pytest.mark.parametrize("where", ["xe", "omega", "chassis", "crank", "controls", "parameters", "all"])
def test_rows_are_the_whole_sweeps(where, value):
    flat = np.ascontiguousarray(params(18, "HMMWV/vehicle.json", "HMMWV/tmeasy.json", False))
    recs, ovr, ctrl = inputs(18, False, flat, 31)
    recs, _ = run(18, False, 1, flat, recs, ovr, ctrl)
    ctl = np.ascontiguousarray(ctrl[-1])
    if where == "controls":
        ctl[0, 2] = ctl[1, 3] = ctl[2, 4] = value
    elif where == "parameters":
        for k in range(N):
            ovr[k, k] = value
    elif where == "all":
        recs[2, :74] = value
    else:
        at = {"xe": [0, 15, 30, 45], "omega": [4, 19, 34, 49], "chassis": [62, 63, 65, 66, 67, 68], "crank": [72]}[where]
        for k in range(N):
            recs[k, at[k % len(at)]] = value
    rows, whole = jacobians(flat, ovr, recs, ctl)
    np.testing.assert_array_equal(rows, whole)
