"""The merit's cuts at the smallest and at coarse grid levels: the fits and the merit changes on them."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


# no 16x16 tile, one tile and its inside, the first levels with nodes above the tiles, 256^2 cells
@pytest.mark.parametrize("level", [2, 3, 4, 5, 8])
def test_cut_sums_match_oracle(level, oracle_mod):
    """The global fit sums over the cut nodes of both cuts, a trial's merit change over those it reaches: relative
    1e-10 and 1e-8, as the suite's other levels."""
    cfg = model.config("composite-4e6", level=level, max_steps=2000000, torbit_fac=1.0)
    w = model.make_workload(cfg, n=1500, target_samples=60000)
    print(f"[gpu] cuts level={level}", flush=True)
    o = oracle_mod.Oracle(w)
    g = GalicGPU(w)
    o.calc_all_response_fields(8)
    g.calc_all_response_fields()
    for t in w.types:
        np.testing.assert_allclose(g.fit(t), o.fit(t), rtol=1e-10)
    idx = model.permutation(w, 1)[:200]
    v = model.trial_velocities(w, idx, 3, 0)
    acc_o, dF_o = o.rep(idx, v, 8)
    acc_g, dF_g = g.rep(idx, v)
    assert np.array_equal(acc_o, acc_g)
    np.testing.assert_allclose(dF_g, dF_o, rtol=1e-8, atol=1e-8 * np.abs(dF_o).max())
    g.close()
    o.close()


@pytest.mark.parametrize("level", [4, 5])
def test_tile_levels_match_whole_grid_merit(level):
    """Form 4 reads a tile's cut levels from its byte, form 2 the weights of every node: the same merit changes to
    form 4's fixed point (at most 1e-4 of the particle's largest change)."""
    cfg = model.config("composite-4e6", level=level, max_steps=2000000, torbit_fac=1.0)
    w = model.make_workload(cfg, n=1500, target_samples=60000)
    idx = model.permutation(w, 2)[:200]
    out = []
    for form in (2, 4):
        g = GalicGPU(w)
        g.fp32_calc_all_response_fields()
        g.fp32_set_merit_form(form)
        g.fp32_rep(idx, k=4, sigma_frac=0.3, seed=7)
        out.append(g.fp32_trial_merits(len(idx), 4))
        g.close()
    scale = np.abs(out[0]).max(axis=1, keepdims=True)
    assert (np.abs(out[1] - out[0]) <= 1e-4 * scale).all()
