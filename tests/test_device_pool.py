"""The buffers of a tree call (galic_pool.h) on the CPU, with an allocator of limited size that keeps its last error
until it is read, as the HIP runtime does."""
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "galic_amd" / "csrc"

HARNESS = r"""
#include <stdio.h>
#include <stdlib.h>
#include <map>
#include "galic_pool.h"

static size_t room, used, peak;
static int last, calls;
static std::map<void *, size_t> live;
struct Mem {
  typedef int Error;
  static int get(void **p, size_t n) {
    calls++;
    if(n > room - used) return last = 2;
    *p = malloc(1);
    live[*p] = n;
    used += n;
    peak = used > peak ? used : peak;
    return 0;
  }
  static void put(void *p) {
    used -= live.at(p);
    live.erase(p);
    free(p);
  }
  static int good() { return 0; }
  static bool is_short(int e) { return e == 2; }
  static void forget() { last = 0; }
};

// argv: room, then the buffers' bytes; prints the result, the last error left, the peak and the allocations
int main(int argc, char **argv) {
  room = strtoull(argv[1], nullptr, 10);
  const int rc = galic::with_pool<galic::DevPool<Mem>>(2, [&](galic::DevPool<Mem> &B) {
    int e = 0;
    for(int i = 2; i < argc && e == 0; i++) {
      char *p = nullptr;
      e = B.alloc(&p, strtoull(argv[i], nullptr, 10));
    }
    return e;
  });
  printf("%d %d %zu %d %zu\n", rc, last, peak, calls, used);
  return 0;
}
"""


def pool(tmp_path, room, sizes):
    exe = tmp_path / "pool"
    if not exe.exists():
        (tmp_path / "pool.cpp").write_text(HARNESS)
        subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(CSRC), str(tmp_path / "pool.cpp"), "-o", str(exe)],
                       check=True)
    out = subprocess.run([str(exe), str(room)] + [str(s) for s in sizes], check=True, capture_output=True, text=True)
    rc, last, peak, calls, used = map(int, out.stdout.split())
    assert used == 0                       # all given back
    return rc, last, peak, calls


MB = 1 << 20


def test_small_calls_share_one_allocation(tmp_path):
    assert pool(tmp_path, 1 << 40, [1000] * 30) == (0, 0, 16 * MB, 1)


def test_a_call_takes_little_more_than_its_buffers(tmp_path):
    sizes = [80 * MB, 80 * MB, 40 * MB, 320 * MB, 40 * MB, 900 * MB, 40 * MB, 11000 * MB, 4000 * MB, 12000 * MB]
    rc, last, peak, calls = pool(tmp_path, 1 << 40, sizes)
    assert (rc, last) == (0, 0) and calls < len(sizes)
    assert peak <= sum(sizes) + 1024 * MB * calls


@pytest.mark.parametrize("spare", [0, 100, 1000])
def test_short_memory_gives_what_fits(tmp_path, spare):
    """Memory for a call's buffers one by one, and less to spare than the room behind them takes: every buffer is had,
    and no error is left behind."""
    sizes = [80 * MB, 40 * MB, 320 * MB, 40 * MB, 900 * MB]
    room = sum(sizes) + spare * MB
    rc, last, peak, _ = pool(tmp_path, room, sizes)
    assert (rc, last) == (0, 0) and peak <= room


def test_memory_that_is_too_short_is_reported_once(tmp_path):
    rc, last, _, _ = pool(tmp_path, 100 * MB, [80 * MB, 40 * MB])
    assert (rc, last) == (2, 0)
