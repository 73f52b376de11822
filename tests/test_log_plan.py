"""The rules that plan the response logs' memory and launches (galic_plan.h), on the CPU."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "galic_amd" / "csrc"

HARNESS = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <vector>
#include "galic_plan.h"

int main(int argc, char **argv) {
  auto arg = [&](int i) { return strtoull(argv[i], nullptr, 10); };
  if(!strcmp(argv[1], "arena")) printf("%d\n", galic::arena_kept(arg(2), arg(3), arg(4), arg(5), arg(6)));
  if(!strcmp(argv[1], "fit"))
    printf("%lld\n", (long long)galic::orbits_fit(atof(argv[2]), atof(argv[3]), atof(argv[4]), atof(argv[5]), atof(argv[6])));
  if(!strcmp(argv[1], "cap")) {
    // the counter of an orbit at the cap after one more step, and whether the kernel's test ends it there
    const long long cap = galic::fp32_step_cap(strtoll(argv[2], nullptr, 10));
    const int steps = (int)(unsigned int)((unsigned long long)cap + 1);
    printf("%lld\n%d\n", cap, steps > 0 && (unsigned int)steps > (unsigned int)cap);
  }
  if(!strcmp(argv[1], "commit")) {
    // the most records of a commit, then the logs' lengths: the runs
    std::vector<int> n;
    for(int i = 3; i < argc; i++) n.push_back(atoi(argv[i]));
    const int m = (int)n.size();
    for(int b0 = 0, run; b0 < m; b0 += run) printf("%d\n", run = galic::commit_run(n.data(), b0, m, atof(argv[2])));
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(CSRC), str(d / "plan.cpp"), "-o", str(d / "plan")],
                   check=True)

    def run(*args):
        out = subprocess.run([str(d / "plan")] + [str(a) for a in args], check=True, capture_output=True, text=True)
        return [int(x) for x in out.stdout.split()]
    return run


# GB: the arena there is, what one launch needs, what the call wants, what holds it in one launch, bounded, kept
@pytest.mark.parametrize("have,need,want,fit,bounded,kept", [
    (0, 1, 10, 9, 0, 0),          # none yet
    (43, 1, 25, 22, 0, 1),        # a second pass after a first one sized with room
    (21, 1, 25, 22, 0, 0),        # one that would need a second launch
    (900, 1, 1000, 897, 0, 1),    # a tenth below what is wanted, and it fits
    (895, 1, 1000, 897, 0, 0),    # 89.5% of what is wanted, and it does not fit: two launches in every call
    (137, 1, 192, 180, 1, 1),     # all the memory wanted, most of it there
    (96, 1, 160, 400, 1, 1),      # a second arena holds the other half
    (75, 1, 160, 400, 1, 0),      # less than half
    (96, 100, 160, 90, 1, 0),     # not one launch's orbits
])
def test_arena_is_kept_unless_a_launch_more_is_saved(plan, have, need, want, fit, bounded, kept):
    gb = 1 << 30
    assert plan("arena", have * gb, need * gb, want * gb, fit * gb, bounded) == [kept]


# arenas of a few blocks to ones far above the full grid's slack (768 workgroups of 256 lanes, 8 blocks each)
@pytest.mark.parametrize("blocks", [3000, 30000, 300000, 1500000, 1600000, 5000000, 40000000])
@pytest.mark.parametrize("per_orbit", [1.06, 10, 75, 300])
def test_orbits_that_fit_leave_room_for_the_slack(plan, blocks, per_orbit):
    """What a launch of that many orbits may need is there, and nearly all of the arena is used: a launch of one
    workgroup more, or of 1% more orbits, would not fit."""
    def needs(m):
        return m * per_orbit + min(-(-m // 256), 768) * 256 * 8
    fit, = plan("fit", blocks, 768 * 256 * 8, 8, 256, per_orbit)
    assert fit >= 1 and needs(fit) <= blocks
    assert needs(fit + max(512, fit // 100)) > blocks


@pytest.mark.parametrize("lengths", [[5], list(range(400, 0, -1)), [900, 3, 3, 3, 800, 1], [0] * 7, [1] * 50 + [700] * 3])
@pytest.mark.parametrize("most", [1, 700, 10000, 1e9])
def test_commit_runs_hold_their_records(plan, lengths, most):
    """Every log once, no commit above its size but for a log alone, none that the next log would still fit in."""
    runs = plan("commit", most, *lengths)
    assert sum(runs) == len(lengths) and min(runs) >= 1
    at = 0
    for r in runs:
        held = sum(lengths[at:at + r])
        assert held <= most or r == 1
        at += r
        assert at == len(lengths) or held + lengths[at] > most


@pytest.mark.parametrize("cap", [1, 100000000, 2**31 - 2, 2**31 - 1])
def test_every_step_cap_ends_an_orbit(plan, cap):
    used, ends = plan("cap", cap)
    assert ends and cap - 1 <= used <= cap
