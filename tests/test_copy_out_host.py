"""Record copies to the host (csrc/copy_out.cpp) on a stand-in for the HIP runtime (tests/cpp/copy_out_check.cpp)."""
import os
import subprocess

import pytest

from conftest import ROOT

CHECK = os.path.join(ROOT, "low-fidelity-dynamic-models_amd", "lfdm_amd", "copy_out_check")


@pytest.mark.parametrize("name", ["per_thread_stream", "waiting_copy_keeps_nothing", "small_reads_apart",
                                  "read_once_pins_nothing", "later_reads_pin_once", "one_cpu", "no_events"])
def test_copy_out(name):
    assert os.path.exists(CHECK), "run make -C low-fidelity-dynamic-models_amd copycheck"
    r = subprocess.run([CHECK, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
