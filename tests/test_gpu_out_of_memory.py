"""A call that asks for more memory than the device has is refused, and nothing else is."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small():
    cfg = model.config("composite-4e6", max_steps=2000000, torbit_fac=0.1)
    w = model.make_workload(cfg, n=2000, target_samples=30000)
    idx = model.permutation(w, 1)[:200]
    return w, idx


def too_much(g):
    """2e8 particles with 64 trials each: their velocities alone are 307 GB."""
    with pytest.raises(RuntimeError, match="out of memory"):
        g.fp32_iterate(np.zeros(200000000, dtype=np.int32), k=64, rep_size=200000000)


def test_refusal_does_not_reach_another_context(small):
    w, idx = small
    a, b = GalicGPU(w), GalicGPU(w)
    a.fp32_calc_all_response_fields()
    too_much(a)
    b.fp32_calc_all_response_fields()
    b.fp32_rep(idx, k=2, sigma_frac=0.1, seed=5)
    a.close()
    b.close()


def test_context_goes_on_after_a_refusal(small):
    """The scratch that the refused call wanted to grow is grown again by the next call."""
    w, idx = small
    acc = []
    for refused in (False, True):
        g = GalicGPU(w)
        g.fp32_calc_all_response_fields()
        first = g.fp32_rep(idx, k=2, sigma_frac=0.1, seed=5)
        if refused:
            too_much(g)
            with pytest.raises(RuntimeError):
                g.fp32_trial_merits(len(idx), 2)
        acc.append((first, g.fp32_rep(idx, k=2, sigma_frac=0.1, seed=6), g.fp32_trial_merits(len(idx), 2)))
        g.close()
    for a, b in zip(*acc):
        assert np.array_equal(a, b)
