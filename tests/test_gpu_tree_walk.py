"""The per-target tree walk, 64 targets on one path: each target's result is that of its own walk."""
import numpy as np
import pytest

from galic_amd import model
from galic_amd.runtime import TREE_FP32, TREE_GROUP, TREE_PLUMMER, TREE_QUADRUPOLE, direct_forces, tree_fill, tree_forces

pytestmark = pytest.mark.gpu


def sources(p, n):
    pos = np.concatenate([model.sample_halo(p, 5, 1, np.arange(n, dtype=np.uint64)),
                          model.sample_halo(p, 5, 2, np.arange(n, dtype=np.uint64), a=p.Bulge_A)])
    mass = np.full(len(pos), 1.0 / len(pos))
    if n > 10:
        pos[7:10] = pos[6]   # a leaf bucket of coincident points
        mass[11] = 0.0       # a source without mass
    return pos, mass


# one target, one short of a wave, a wave, one more, many waves in Morton order
@pytest.mark.parametrize("ntarget", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("mode", [0, TREE_FP32, TREE_QUADRUPOLE, TREE_FP32 | TREE_QUADRUPOLE | TREE_PLUMMER])
def test_each_target_walks_for_itself(mode, ntarget):
    p = model.make_params(model.config("composite-4e6"))
    pos, mass = sources(p, 1500)
    t = 0.5 * pos[np.arange(ntarget) * 3 % len(pos)]   # inside the sources' extent: the same domain cube for any subset
    print(f"[gpu] walk mode={mode} ntarget={ntarget}", flush=True)
    acc, pot, nint = tree_forces(p, pos, mass, t, precision=mode)
    total = 0
    picks = np.arange(ntarget) if ntarget <= 65 else np.array([0, 1, 500, 998, 999])
    for k in picks:
        a1, p1, n1 = tree_forces(p, pos, mass, t[k:k + 1], precision=mode)
        assert np.array_equal(acc[k], a1[0]) and pot[k] == p1[0], k
        total += n1
    if ntarget <= 65:
        assert total == nint


@pytest.mark.parametrize("nsrc", [0, 1, 2, 9])
def test_few_sources_equal_direct_summation(nsrc):
    """Down to no source at all, theta -> 0: every source on its own, FP64 to 1e-12."""
    p = model.make_params(model.config("composite-4e6", theta=1e-6))
    pos, mass = sources(p, 10)
    pos, mass = pos[:nsrc], mass[:nsrc]
    t = model.sample_halo(p, 6, 3, np.arange(70, dtype=np.uint64))
    acc, pot, nint = tree_forces(p, pos, mass, t)
    assert nint == 70 * nsrc
    if nsrc:
        da, dp = direct_forces(p, pos, mass, t)
        np.testing.assert_allclose(acc, da, rtol=1e-12, atol=1e-12 * np.abs(da).max())
        np.testing.assert_allclose(pot, dp, rtol=1e-12)
    else:
        assert not acc.any() and not pot.any()


# list lengths around the batch of four, a bucket (from 12 sources on), several flushes of a list
@pytest.mark.parametrize("nsrc", [1, 3, 4, 5, 8, 12, 13, 64, 2999])
def test_group_lists_of_any_length_equal_direct_summation(nsrc):
    """theta -> 0: the group's list holds every source.  A term's FP32 chain (difference, r^2, two
    reciprocal roots, products) is within 32 roundings, a sum of n terms within n more: each
    component within (32 + n) 2^-24 of the sum of its terms' magnitudes."""
    p = model.make_params(model.config("composite-4e6", theta=1e-6))
    pos, mass = sources(p, 1500)
    pos, mass = pos[:nsrc], mass[:nsrc]
    t = model.sample_halo(p, 6, 3, np.arange(70, dtype=np.uint64))
    print(f"[gpu] group list nsrc={nsrc}", flush=True)
    acc, pot, nint = tree_forces(p, pos, mass, t, precision=TREE_FP32 | TREE_PLUMMER | TREE_GROUP)
    assert nint == 70 * np.count_nonzero(mass)
    da, dp = direct_forces(p, pos, mass, t, plummer=True)
    d = pos[None] - t[:, None]
    r = np.sqrt((d ** 2).sum(axis=2))
    tol = (32 + nsrc) * 2.0 ** -24
    scale = p.G * (mass[None, :, None] * np.abs(d) / np.maximum(r, 1e-300)[..., None] ** 3).sum(axis=1)
    assert (np.abs(acc - da) <= tol * scale).all()
    assert (np.abs(pot - dp) <= tol * np.abs(dp)).all()


def count_interactions(pos, mass, t, theta, depth=21):
    """An octree of its own: the interactions of every target's walk."""
    both = np.concatenate([pos, t])
    lo, hi = both.min(axis=0), both.max(axis=0)
    size = (hi - lo).max() * 1.00001
    key = np.floor((pos - 0.5 * (lo + hi) + 0.5 * size) / size * 2 ** depth).astype(np.int64)

    def node(idx, d, tt, width):
        if len(idx) == 1:
            return len(tt)
        com = mass[idx] @ pos[idx] / mass[idx].sum()
        opened = np.float32(width * width) > ((com - t[tt]) ** 2).sum(axis=1) * theta * theta
        n, tt = np.count_nonzero(~opened), tt[opened]
        if len(tt) == 0 or d == depth:
            return n + len(tt) * len(idx)
        octant = ((key[idx] >> (depth - 1 - d)) & 1) @ np.array([1, 2, 4])
        return n + sum(node(idx[octant == k], d + 1, tt, width / 2) for k in set(octant))

    return node(np.arange(len(pos)), 0, np.arange(len(t)), size)


# a workgroup's 128 nodes of a level: fewer, as many, one more; deep chains (pairs closer than a node)
@pytest.mark.parametrize("npair", [1, 127, 128, 129, 1025])
def test_tree_of_close_pairs_equals_direct_summation(npair):
    """Pairs far closer than their distance to the next pair: every pair a node of its own on many
    levels; theta -> 0, FP64 to 1e-12 (a pair smaller than 1e-6 of its distance counts once)."""
    p = model.make_params(model.config("composite-4e6", theta=1e-6))
    c = model.sample_halo(p, 7, 1, np.arange(npair, dtype=np.uint64))
    pos = np.concatenate([c, c * (1 + 1e-5)])
    mass = np.linspace(0.5, 1.5, len(pos)) / len(pos)
    t = model.sample_halo(p, 7, 3, np.arange(70, dtype=np.uint64))
    print(f"[gpu] tree of {npair} pairs", flush=True)
    acc, pot, nint = tree_forces(p, pos, mass, t)
    assert nint == count_interactions(pos, mass, t, p.ErrTolTheta)
    da, dp = direct_forces(p, pos, mass, t)
    np.testing.assert_allclose(acc, da, rtol=1e-12, atol=1e-12 * np.abs(da).max())
    np.testing.assert_allclose(pot, dp, rtol=1e-12)


# one target a wave up to 2047; two, four, 32, 64 from there on (the first and last count of each)
@pytest.mark.parametrize("ntarget", [2047, 2048, 4097, 65535, 65537])
@pytest.mark.parametrize("mode", [0, TREE_FP32 | TREE_QUADRUPOLE | TREE_PLUMMER])
def test_targets_do_not_depend_on_their_wave(mode, ntarget):
    p = model.make_params(model.config("composite-4e6"))
    pos, mass = sources(p, 1500)
    rng = np.random.default_rng(ntarget)
    t = pos[rng.integers(0, len(pos), ntarget)] * rng.uniform(0.1, 0.9, (ntarget, 1))   # the domain cube is the sources'
    print(f"[gpu] targets a wave mode={mode} ntarget={ntarget}", flush=True)
    acc, pot, _ = tree_forces(p, pos, mass, t, precision=mode)
    pick = np.unique(np.concatenate([np.arange(70), ntarget - 1 - np.arange(70), rng.integers(0, ntarget, 300)]))
    a1, p1, _ = tree_forces(p, pos, mass, t[pick], precision=mode)
    assert np.array_equal(acc[pick], a1) and np.array_equal(pot[pick], p1)


# waves of 1, 2, 4, 8 and 32 table nodes of an 8 x 8 block
@pytest.mark.parametrize("nb", [8, 16, 24, 32, 64])
def test_small_fill_equals_forces_at_its_nodes(nb):
    """The nodes' places differ by the rounding of cos and sin, the sums over sections by theirs: 1e-12."""
    p = model.make_params(model.config("composite-4e6", fg_nbin=nb))
    pos, mass = sources(p, 1500)
    pot, dr, dz, n = tree_fill(p, pos, mass)
    phi = 2 * np.pi / 8 * np.arange(8)
    r = p.FG_Rmin * (p.FG_Fac ** np.arange(nb) - 1.0)
    s, k, j = np.meshgrid(np.arange(8), np.arange(nb), np.arange(nb), indexing="ij")
    t = np.stack([r[j] * np.cos(phi[s]), r[j] * np.sin(phi[s]), r[k]], axis=-1).reshape(-1, 3)
    acc, pt, nf = tree_forces(p, pos, mass, t)
    assert nf == n
    acc, pt = acc.reshape(8, nb * nb, 3), pt.reshape(8, nb * nb)
    np.testing.assert_allclose(pot, pt.mean(axis=0), rtol=1e-12)
    rad = acc[:, :, 0] * np.cos(phi)[:, None] + acc[:, :, 1] * np.sin(phi)[:, None]
    scale = np.abs(acc).max(axis=(0, 2))
    assert (np.abs(dr - rad.mean(axis=0)) <= 1e-12 * scale).all()
    assert (np.abs(dz - acc[:, :, 2].mean(axis=0)) <= 1e-12 * scale).all()
