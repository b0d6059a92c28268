"""Header-only host routines of the library, compiled by themselves and run on
the CPU: how the waves of a persistent ray batch share its rays
(work_slices.h), and loops on several threads (parallel_for.h)."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bling_amd", "csrc")


def _run(tmp_path, source, *args):
    src, exe = str(tmp_path / "t.cpp"), str(tmp_path / "t")
    with open(src, "w") as f:
        f.write(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + CSRC, src, "-o", exe, "-ldl", "-lpthread"], check=True)
    return subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=60)


SLICES = """
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "work_slices.h"
using namespace bgpu;
// Blocks of two waves take slices in turn until their counters run out, with
// the library's counters or (planted) with 16 of them whatever the grid.
static bool covered(unsigned n, unsigned blocks, bool planted) {
  const unsigned slice = slice_items(n, 2 * blocks, 128);
  std::vector<unsigned> counter(kWorkCounters, 0), taken(n, 0);
  std::vector<char> drained(2 * blocks, 0);
  for (unsigned left = 2 * blocks; left;)
    for (unsigned w = 0; w < 2 * blocks; ++w) {
      if (drained[w]) continue;
      const unsigned b = w / 2, own = planted ? b % kWorkCounters : counter_of(b, blocks);
      if (own >= kWorkCounters) return false;
      const unsigned k = counter[own]++;
      const unsigned long long base =
          planted ? ((unsigned long long)k * kWorkCounters + own) * slice : slice_begin(k, b, blocks, slice);
      if (base >= n) { drained[w] = 1; --left; continue; }
      for (unsigned long long i = base; i < base + slice && i < n; ++i) ++taken[i];
    }
  for (unsigned t : taken)
    if (t != 1) return false;
  return true;
}
int main() {
  for (unsigned blocks : {1u, 2u, 5u, 15u, 16u, 17u, 31u, 240u, 3072u})
    for (unsigned n : {1u, 63u, 64u, 65u, 1023u, 1025u, 4096u, 100003u, 1572863u, 1572864u, 2000003u})
      if (!covered(n, blocks, false)) return printf("%u items, %u blocks\\n", n, blocks), 1;
  return covered(100003, 15, true) || !covered(100003, 16, true) ? 2 : 0;
}
"""


def test_every_slice_has_a_block(tmp_path):
    """Each ray is taken exactly once on every grid, also one of fewer blocks
    than counters (the planted rule, which gives a counter no block there,
    leaves rays out)."""
    r = _run(tmp_path, SLICES)
    assert r.returncode == 0, r.stdout


THREADS = """
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <cstdio>
#include <cstdlib>
#include "parallel_for.h"
static int allowed;
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* p) {
  static auto real = (decltype(&pthread_create))dlsym(RTLD_NEXT, "pthread_create");
  return allowed-- > 0 ? real(t, a, f, p) : EAGAIN;
}
int main(int, char** argv) {
  allowed = atoi(argv[1]);
  std::vector<int> seen(1000003, 0);
  bgpu::parallel_for(seen.size(), [&](size_t b, size_t e) { for (size_t i = b; i < e; ++i) ++seen[i]; });
  for (int s : seen)
    if (s != 1) return 1;
  return 0;
}
"""


@pytest.mark.parametrize("threads", [0, 1, 100])
def test_loop_without_threads_to_start(tmp_path, threads):
    """A system that grants no (further) thread gets the whole loop done, not
    an exception through the C interface."""
    r = _run(tmp_path, THREADS, threads)
    assert r.returncode == 0, r.stderr
