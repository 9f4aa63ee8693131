"""The reverse sweep's lanes on the storage its kernel gives them (ReverseStore, csrc/d18_group_adjoint.h).  Every
lane runs as a thread here (tests/cpp/group_step.cpp) and the lanes are not in step, so adjoints that several of
them added to would come out wrong."""
import ctypes

import numpy as np
import pytest

from test_group_host import LIB, N, inputs, params


@pytest.mark.parametrize("lanes", [2, 4])
@pytest.mark.parametrize("veh", ["HMMWV", "audi"])
def test_lanes_out_of_step_give_the_one_lane_bits(veh, lanes):
    steps, K = 60, 60
    flat = np.ascontiguousarray(params(18, f"{veh}/vehicle.json", f"{veh}/tmeasy.json", False))
    recs, ovr, ctrl = inputs(18, False, flat, 78)
    ctrl = np.ascontiguousarray(ctrl[:steps])
    xy_bar = np.random.Generator(np.random.PCG64(6)).normal(size=(steps, 2, N))
    L = ctypes.CDLL(LIB)
    i, p = ctypes.c_int, ctypes.c_void_p
    L.group_adjoint_run.argtypes = [i, p, i, p, p, i, i, i, i, p, p, p, p, p, p]

    def gradients(lanes):
        out = [np.zeros((steps, 2, N)), np.zeros((steps, 3, N)), np.zeros((75, N)), np.zeros((7, N))]
        assert L.group_adjoint_run(lanes, flat.ctypes.data, flat.size, ovr.ctypes.data, recs.ctypes.data, N, steps, K,
                                   1, ctrl.ctypes.data, xy_bar.ctypes.data, *[a.ctypes.data for a in out]) == 0
        return out

    for name, a, b in zip(("xy", "controls", "record", "parameters"), gradients(-lanes), gradients(1)):
        np.testing.assert_array_equal(a, b, err_msg=name)
