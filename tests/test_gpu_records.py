"""Records read back from the GPU (lfdm_get_states) through each of its ways: gathered into pinned memory
(up to 1 MiB), copied plainly, and by several threads through pinned parts of 2 MiB (from 4 MiB on)."""
import threading
import time

import numpy as np
import pytest

import lfdm_amd
from lfdm_amd import workloads as W
from lfdm_amd._lib import check, lib
from lfdm_amd.solver import SolverHalfImplicitGPU, TMeasy

pytestmark = pytest.mark.gpu

REC = 75 * 8
MIB = 1 << 20


def fleet(n, seed):
    flat = lfdm_amd.params_from_json(18, W.HMMWV_VEH, W.HMMWV_TIRE)
    recs = np.random.Generator(np.random.PCG64(seed)).normal(size=(n, 75))
    s = SolverHalfImplicitGPU(18, n)
    s.construct_flat(flat, n, None, TMeasy)
    s.Initialize(s.zero_record(), n)
    return s, recs


def on_device(s, recs):
    import torch

    t = torch.from_numpy(recs).cuda()
    torch.cuda.synchronize()
    s.set_states_device(t.data_ptr())
    s.synchronize()
    return t


# around 1 MiB, 4 MiB, and parts of 2 MiB: one per thread and one more, with a remainder
SIZES = [1, MIB // REC, MIB // REC + 1, 4 * MIB // REC, 4 * MIB // REC + 1, 32 * MIB // REC, 33 * MIB // REC + 7,
         100_003]


@pytest.mark.parametrize("n", SIZES)
def test_records_come_back_whole(n):
    import torch

    s, recs = fleet(n, n)
    on_device(s, recs)
    for _ in range(2):
        np.testing.assert_array_equal(s.get_states(), recs)
    pinned = torch.empty((n, 75), dtype=torch.float64, pin_memory=True)
    check(lib.lfdm_get_states(s._h, pinned.data_ptr()))
    np.testing.assert_array_equal(pinned.numpy(), recs)
    s.close()


def test_several_fleets_read_back_at_once():
    fleets = [fleet(n, n) for n in (40_000, 1_000, 30_000, 1_500)]
    for s, recs in fleets:
        on_device(s, recs)
    wrong = []

    def read(s, recs):
        for _ in range(20):
            if not np.array_equal(s.get_states(), recs):
                wrong.append(recs.shape)

    threads = [threading.Thread(target=read, args=x) for x in fleets]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for s, _ in fleets:
        s.close()


def test_handles_come_and_go_while_another_reads_back():
    """A read back waits for the work ahead of it (some 1 s here); a handle made meanwhile does not."""
    flat = lfdm_amd.params_from_json(18, W.HMMWV_VEH, W.HMMWV_TIRE)
    s = SolverHalfImplicitGPU(18, 64)
    s.construct_flat(flat, 64, np.array([[0.0, 0.0, 0.2, 0.0], [1.0, 0.0, 0.2, 0.0]]), TMeasy)
    s.Initialize(s.zero_record(), 64)
    s.set_controls_table()
    s.advance(10)
    s.get_states()
    s.advance(400_000)
    reader = threading.Thread(target=s.get_states)
    reader.start()
    time.sleep(0.05)
    SolverHalfImplicitGPU(11, 1).close()
    still_reading = reader.is_alive()
    reader.join()
    s.close()
    assert still_reading
