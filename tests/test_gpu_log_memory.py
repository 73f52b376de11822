"""The FP32 path's response logs: how much memory they have does not show in the results, and is not taken anew by
the next call."""
import ctypes

import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


def free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.fixture(scope="module")
def full():
    """The full model's grids, where the estimate from the orbits' start points is lowest."""
    cfg = model.config("composite-2e7", max_steps=2000000)
    return model.make_workload(cfg, n=4000, target_samples=100000)


def test_second_pass_takes_no_memory(full):
    g = GalicGPU(full)
    g.fp32_calc_all_response_fields()
    assert g.timings()["log_relaunches"] <= 1   # (a log longer than the block tables held)
    before = free_bytes()
    g.fp32_calc_all_response_fields()
    assert abs(free_bytes() - before) < 64 << 20
    assert g.timings()["orbit_launches"] == 2
    g.close()
