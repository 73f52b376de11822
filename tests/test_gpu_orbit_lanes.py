"""Orbits spread over the lanes of a launch: the results do not depend on how many orbits share it."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def composite():
    """All three components; a short integration so that launches of many orbits stay quick."""
    cfg = model.config("composite-4e6", max_steps=2000000, torbit_fac=0.2)
    return model.make_workload(cfg, n=3000, target_samples=100000)


# one quad a wave, four, a partly filled last wave, waves of 16 quads, more orbits than resident quads (sorted)
@pytest.mark.parametrize("n", [1, 3, 257, 1030, 16 * 1024 + 5, 50001])
def test_fp64_orbits_do_not_depend_on_the_launch(composite, oracle_mod, n):
    w = composite
    print(f"[gpu] fp64 orbits n={n}", flush=True)
    i = np.arange(n) % w.n
    g = GalicGPU(w)
    r = g.orbit_responses(w.pos[i], w.vel[i], w.mass[i], w.tint[i], w.ptype[i], fields=False)
    pick = np.unique(np.concatenate([np.arange(min(n, 3)), [n // 2, n - 1]]))
    o = oracle_mod.Oracle(w, set_particles=False)
    for k in pick:
        j = i[k]
        one = g.orbit_responses(w.pos[j], w.vel[j], w.mass[j], w.tint[j], w.ptype[j])
        ro = o.orbit(w.pos[j], w.vel[j], w.mass[j], w.tint[j], w.ptype[j])
        for key in ("t", "orbits", "steps", "e0", "e1"):
            assert r[key][k] == one[key][0], (n, k, key)
        assert one["steps"][0] == ro["steps"] and one["orbits"][0] == ro["orbits"]
        rel = np.abs(one["fields"][0] - ro["fields"]).sum(axis=1) / np.abs(ro["fields"]).sum(axis=1)
        assert (rel <= 1e-10).all(), (n, k, rel)
    g.close()
    o.close()


def test_fp64_initial_pass_sorted(composite):
    """An initial pass of more particles than resident quads (longest expected first): every orbit is counted once
    (the mass field's total is the component's mass) and its result is written to its own particle."""
    cfg = model.config("halo-1e5", max_steps=2000000, torbit_fac=0.1)
    w = model.make_workload(cfg, n=50001, target_samples=100000)
    g = GalicGPU(w)
    g.calc_all_response_fields()
    orbits = g.particles()[1]
    r = g.orbit_responses(w.pos, w.vel, w.mass, w.tint, w.ptype, fields=False)
    assert np.array_equal(orbits, r["orbits"])
    assert g.stack(1, 0)[0] == pytest.approx(w.params.MType[1], rel=1e-12)
    g.close()
