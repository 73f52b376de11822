"""How the sampled targets are split into launches does not show: maps against the oracle's binning of
the same points on both sides of the rule's lines, and points of a stretched halo against host draws."""
import numpy as np
import pytest

from galic_amd import model, rng
from galic_amd.runtime import GalicGPU

pytestmark = pytest.mark.gpu


# maps of 8, 32 and 128 KiB; the last sample count with small workgroups and the first with large ones
@pytest.mark.parametrize("n", [1, 65535, 65536])
@pytest.mark.parametrize("level", [5, 6, 7])
def test_maps_equal_binned_points(level, n, oracle_mod):
    """A weight is rounded to 2^-32, so a mass map is within n/2 units of it: 2^-33 of the mass."""
    w = model.make_workload(model.config("composite-4e6", level=level), n=4000, target_samples=1000)
    p = w.params
    g = GalicGPU(w)
    o = oracle_mod.Oracle(w, set_particles=False)
    try:
        beta, tabs = model.disp_tables(p, w.cfg, 1)
        g.set_disp_tables(1, beta, **tabs)
        o.set_disp_tables(1, beta, **tabs)
        print(f"[gpu] targets level={level} n={n}", flush=True)
        dg, eg, nb, _, pts = g.sample_targets(1, n, seed=4, points=True)
        rdg, reg, rn = o.bin_targets(1, pts)
        assert nb == rn
        assert np.abs(dg - rdg).max() <= 1e-9 * p.MType[1]
        assert np.abs(eg[0] - reg[0]).max() <= 1e-9 * p.MType[1]
        only_dg = g.sample_targets(1, n, seed=4, energy=False)
        only_eg = g.sample_targets(1, n, seed=4, density=False)
        assert np.array_equal(only_dg[0], dg) and np.array_equal(only_eg[1], eg)
    finally:
        o.close()
        g.close()


@pytest.mark.parametrize("level", [5, 6, 7])
def test_one_more_point_changes_its_own_cells_only(level):
    """65535 points and 65536 are summed by different launches.  The sums are whole numbers, so the
    maps differ in the last point's four cells; elsewhere only by the normalisation's three roundings,
    taken twice: 8 2^-53 of the value."""
    w = model.make_workload(model.config("composite-4e6", level=level), n=4000, target_samples=1000)
    p = w.params
    g = GalicGPU(w)
    try:
        beta, tabs = model.disp_tables(p, w.cfg, 1)
        g.set_disp_tables(1, beta, **tabs)
        off = model.stack_offset(p.DG_MaxLevel, 0, 0)
        print(f"[gpu] targets level={level} one more point", flush=True)
        a, b = (g.sample_targets(1, n, seed=4) for n in (65535, 65536))
        sa, sb = a[1][:, off:] * a[2], b[1][:, off:] * b[2]
        differ = np.abs(sa - sb) > 8 * 2.0 ** -53 * np.abs(sb)
        assert (differ.sum(axis=1) <= 4).all()
        assert b[2] - a[2] == differ.any()
        assert np.array_equal(np.flatnonzero(differ.any(axis=0)), np.flatnonzero(differ[0]))
    finally:
        g.close()


@pytest.mark.parametrize("t", [1, 3])
@pytest.mark.parametrize("stretch", [0.5, 2.0])
def test_stretched_points_equal_host_draws(t, stretch, oracle_mod):
    """Radii beyond the grid whose stretched point is inside it are kept, and the others drawn again."""
    w = model.make_workload(model.config("composite-4e6"), n=4000, target_samples=1000)
    p = w.params
    g = GalicGPU(w)
    try:
        n = 20000
        print(f"[gpu] points type={t} stretch={stretch}", flush=True)
        _, _, _, _, pts = g.sample_targets(t, n, seed=9, stream=200 + t, stretch=stretch, energy=False, points=True)
        ref = oracle_mod.sample_points(p, t, np.arange(n, dtype=np.uint64), rng.uniforms, 9, 200 + t, stretch=stretch)
        np.testing.assert_allclose(pts, ref, rtol=1e-12, atol=1e-13 * p.Rmax)
    finally:
        g.close()
