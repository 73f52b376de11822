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


def state(g, types):
    """Every grid the particles' responses add up to, their pericentre counts and velocities, and the fits."""
    vel, orbits, _ = g.particles()
    return [g.stack(t, k) for t in types for k in range(10)] + [g.fit(t) for t in types] + [vel, orbits]


def assert_same(a, b):
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.fixture(scope="module")
def one_share(full):
    g = GalicGPU(full)
    g.fp32_calc_all_response_fields()
    ref = state(g, full.types)
    g.close()
    return ref


# logs of 1.5 GB in several shares, each committed at once; in one, committed in many runs; both
@pytest.mark.parametrize("log_mb,commit_mb", [(600, 0), (0, 8), (400, 8)])
def test_initial_pass_in_parts(full, one_share, log_mb, commit_mb):
    """Sums of whole numbers: the same bits however the orbits are shared out."""
    g = GalicGPU(full)
    g.fp32_set_memory(log_mb << 20, commit_mb << 20)
    print(f"[gpu] initial pass, logs {log_mb} MB, commits {commit_mb} MB", flush=True)
    g.fp32_calc_all_response_fields()
    assert (g.timings()["orbit_launches"] > 1) == (log_mb > 0)
    assert_same(state(g, full.types), one_share)
    g.close()


@pytest.mark.parametrize("log_mb", [0, 600])
def test_initial_pass_planned_on_short_orbits(full, one_share, log_mb):
    """A pass of orbits a twentieth as long sets the estimate for the next: its launch runs out of arena and its
    shares are halved, then divided by the corrected estimate."""
    tint = full.tint.copy()
    g = GalicGPU(full)
    g.fp32_set_memory(log_mb << 20)
    full.tint[:] = tint / 20
    g.set_particles(full.pos, full.vel)
    full.tint[:] = tint
    g.fp32_calc_all_response_fields()
    g.set_particles(full.pos, full.vel)
    g.set_dispersions(full.disp)
    g.reset_timings()
    print(f"[gpu] initial pass planned on short orbits, logs {log_mb} MB", flush=True)
    g.fp32_calc_all_response_fields()
    t = g.timings()
    assert t["log_relaunches"] >= 1 and t["orbit_launches"] >= 3
    assert_same(state(g, full.types), one_share)
    g.close()


@pytest.mark.parametrize("overlap", [0, 1])
def test_reps_planned_on_short_orbits(full, overlap):
    """Reps of the shortest orbits set the estimate for those of the longest, whose launch runs out of arena: the
    group is planned again, smaller, with the same trials and the same results."""
    g = GalicGPU(full)
    steps = g.orbit_responses(full.pos, full.vel, full.mass, full.tint, full.ptype, fields=False, precision=32)["steps"]
    g.close()
    order = np.argsort(steps)
    out, launches = [], []
    for log_mb in (0, 400):
        g = GalicGPU(full)
        g.fp32_calc_all_response_fields()
        g.fp32_set_memory(log_mb << 20)
        g.fp32_set_schedule(overlap=overlap)
        acc = [g.fp32_rep(order[:200], k=4, sigma_frac=0.1, seed=3)]
        g.reset_timings()
        print(f"[gpu] reps planned on short orbits, logs {log_mb} MB, overlap {overlap}", flush=True)
        acc.append(g.fp32_iterate(order[-900:], k=4, rep_size=450, sigma_frac=0.1, seed=4))
        t = g.timings()
        launches.append(t["orbit_launches"])
        assert log_mb == 0 or t["log_relaunches"] >= 1
        out.append(acc + state(g, full.types))
        g.close()
    assert launches[1] > launches[0]
    assert_same(*out)


def test_memory_bound_holds_after_larger_arenas(full, one_share):
    """Two arenas of an overlapped schedule give way when the caller bounds the logs."""
    g = GalicGPU(full)
    g.fp32_calc_all_response_fields()
    first = free_bytes()
    g.fp32_set_memory(400 << 20)
    g.fp32_calc_all_response_fields()
    assert free_bytes() > first + (1 << 30)     # an arena of 2 GB and more gave way to one of 400 MB
    g.fp32_set_schedule(overlap=1)
    g.fp32_rep(np.arange(100), k=2, sigma_frac=0.1, seed=3)
    g.fp32_set_schedule(overlap=0)
    g.fp32_set_memory(150 << 20)
    g.set_particles(full.pos, full.vel)
    g.set_dispersions(full.disp)
    g.reset_timings()
    g.fp32_calc_all_response_fields()
    assert g.timings()["orbit_launches"] < 50
    assert_same(state(g, full.types), one_share)
    with pytest.raises(RuntimeError):
        g.fp32_set_memory(1000)
    g.close()
