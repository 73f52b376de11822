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


# one lane, a full wave and one more, a full workgroup and one more, more orbits than resident lanes
@pytest.mark.parametrize("n", [1, 64, 65, 257, 300001])
def test_fp32_orbits_do_not_depend_on_the_launch(n):
    """Batched FP32 orbits equal the same orbits integrated alone, bit for bit, and follow the FP64 path: the energies
    at the start to rounding, the mass response of every orbit sums to its particle's mass (FP32 sums of some hundred
    records: 1e-4)."""
    cfg = model.config("composite-4e6", max_steps=2000000, torbit_fac=0.05, level=4)
    w = model.make_workload(cfg, n=2000, target_samples=20000)
    print(f"[gpu] fp32 orbits n={n}", flush=True)
    i = np.arange(n) % w.n
    g = GalicGPU(w)
    few = n <= 257
    r = g.orbit_responses(w.pos[i], w.vel[i], w.mass[i], w.tint[i], w.ptype[i], fields=few, precision=32)
    for k in np.unique([0, n // 3, n // 2, n - 1]):
        j = i[k]
        one = g.orbit_responses(w.pos[j], w.vel[j], w.mass[j], w.tint[j], w.ptype[j], precision=32)
        for key in ("t", "orbits", "steps", "e0", "e1") + (("fields",) if few else ()):
            assert np.array_equal(r[key][k], one[key][0]), (n, k, key)
        assert one["fields"][0][0].sum() == pytest.approx(w.mass[j], rel=1e-4)
        assert one["e0"][0] == pytest.approx(g.orbit_responses(w.pos[j], w.vel[j], w.mass[j], w.tint[j], w.ptype[j],
                                                              fields=False)["e0"][0], rel=1e-12)
    g.close()
