"""The 16 x 16-tile merit: trial counts on both sides of the kernel variants' limits, from one particle to many."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n", [1, 8, 9, 150])
def test_every_trial_count_matches_whole_grid_merit(k, n):
    """Form 4 rounds a record's value to 2^-31 of the particle's largest total, form 2 does not: merit changes
    within 1e-4 of the particle's largest (a sum over thousands of records and nodes)."""
    cfg = model.config("composite-4e6", max_steps=2000000, torbit_fac=1.0)
    w = model.make_workload(cfg, n=1500, target_samples=60000)
    idx = model.permutation(w, 2)[:n]
    print(f"[gpu] merit parts k={k} n={n}", flush=True)
    out = []
    for form in (2, 4):
        g = GalicGPU(w)
        g.fp32_calc_all_response_fields()
        g.fp32_set_merit_form(form)
        acc = g.fp32_rep(idx, k=k, sigma_frac=0.3, seed=7)
        dfk = g.fp32_trial_merits(n, k)
        best = np.where(dfk.min(axis=1) < 0, dfk.argmin(axis=1) + 1, 0)
        assert np.array_equal(acc, best)
        out.append(dfk)
        g.close()
    scale = np.abs(out[0]).max(axis=1, keepdims=True)
    assert (np.abs(out[1] - out[0]) <= 1e-4 * scale).all()
