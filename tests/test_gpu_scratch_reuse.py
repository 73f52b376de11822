"""Scratch memory that calls share: what one call leaves in it does not reach the next one's results."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def small():
    cfg = model.config("composite-4e6", max_steps=2000000, torbit_fac=0.3)
    w = model.make_workload(cfg, n=3000, target_samples=60000)
    idx = model.permutation(w, 1)[:300]
    g = GalicGPU(w)
    g.calc_all_response_fields()
    v = model.trial_velocities(w, idx, 3, 0)
    ref = g.rep(idx, v)
    g.close()
    return w, idx, v, ref


def same_rep(g, idx, v, ref):
    """The initial pass sums with FP64 atomics in any order, the orbits are the same: merit changes to 1e-8 of the
    largest, as between two contexts that do nothing else."""
    acc, dF = g.rep(idx, v)
    assert np.array_equal(acc, ref[0])
    np.testing.assert_allclose(dF, ref[1], rtol=1e-8, atol=1e-8 * np.abs(ref[1]).max())


def test_fp64_rep_after_response_logs(small):
    """The FP32 path's response logs and the FP64 path's orbit slots share one buffer."""
    w, idx, v, ref = small
    g = GalicGPU(w)
    g.fp32_calc_all_response_fields()
    g.fp32_rep(idx, k=2, sigma_frac=0.1, seed=5)
    g.set_particles(w.pos, w.vel)
    g.set_dispersions(w.disp)
    g.calc_all_response_fields()
    same_rep(g, idx, v, ref)
    g.close()


@pytest.mark.parametrize("precision", [32, 64])
def test_fp64_rep_after_orbit_fields(small, precision):
    w, idx, v, ref = small
    g = GalicGPU(w)
    i = np.arange(700) % w.n
    g.orbit_responses(w.pos[i], w.vel[i], w.mass[i], w.tint[i], w.ptype[i], precision=precision)
    g.calc_all_response_fields()
    same_rep(g, idx, v, ref)
    g.close()


def test_fp64_rep_after_orbits_that_failed(small):
    """Orbits integrated without fields bin into the rep's delta grids; one beyond the step cap ends the call early."""
    w, idx, v, ref = small
    cap = w.params.MaxStepsPerOrbit
    w.params.MaxStepsPerOrbit = 20000
    g = GalicGPU(w)
    w.params.MaxStepsPerOrbit = cap
    g.calc_all_response_fields()
    with pytest.raises(RuntimeError, match="step cap"):
        g.orbit_responses(w.pos[:50], w.vel[:50], w.mass[:50], 1000 * w.tint[:50], w.ptype[:50], fields=False)
    same_rep(g, idx, v, ref)
    # an accepted orbit takes the place of one of the same mass: sums of 3000 orbits, 1e-10
    for t in w.types:
        assert g.stack(t, 0)[0] == pytest.approx(w.params.MType[t], rel=1e-10)
    g.close()
