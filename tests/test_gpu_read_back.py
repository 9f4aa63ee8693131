"""Records read back (lfdm_get_states) on streams of the caller's."""
import numpy as np
import pytest

import lfdm_amd
from lfdm_amd import workloads as W
from lfdm_amd.solver import SolverHalfImplicitGPU, TMeasy

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread: a handle value that names another stream in every thread


def fleet(n, stream=None):
    flat = lfdm_amd.params_from_json(18, W.HMMWV_VEH, W.HMMWV_TIRE)
    s = SolverHalfImplicitGPU(18, n)
    if stream is not None:
        s.set_stream(stream)
    s.construct_flat(flat, n, np.array([[0.0, 0.0, 0.2, 0.0], [1.0, 0.3, 0.5, 0.0]]), TMeasy)
    s.Initialize(s.zero_record(), n)
    s.set_controls_table()
    return s


@pytest.mark.parametrize("n", [64, 100_003])
def test_records_follow_the_work_of_a_per_thread_stream(n):
    """Every vehicle has the state after the steps asked for, though they are pending when the read back starts."""
    ref = fleet(n)
    s = fleet(n, PER_THREAD)
    for _ in range(3):
        ref.advance(2000)
        ref.synchronize()
        s.advance(2000)
        np.testing.assert_array_equal(s.get_states(), ref.get_states())
    ref.close()
    s.close()
