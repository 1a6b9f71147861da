"""parallel_for (taurus_vap_amd/csrc/tg_parallel.h), the threads of tg_init, when memory runs
out: in starting a thread (the others take its share and every item is done), before the
first one or in an item (std::bad_alloc, which tg_init returns as TG_E_NOMEM).  A host
program whose operator new fails at the k-th allocation of its first thread; ending by
anything but a return is a failure."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "taurus_vap_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "tg_parallel.h"
static thread_local int left = 0;        // the allocation that fails (0: none)
void* operator new(std::size_t n) {
  if (left > 0 && --left == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
int main(int, char** argv) {
  const int k = std::atoi(argv[1]), item = std::atoi(argv[2]);
  std::atomic<int> done(0);
  left = k;
  try {
    parallel_for<int>(200, 8, [&](int g, int&) {
      if (g == item) throw std::bad_alloc();
      ++done;
    });
    std::printf("done %d\n", (int)done);
  } catch (const std::bad_alloc&) {
    std::printf("bad_alloc\n");
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("parallel")
    src, exe = d / "p.cpp", d / "p"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    return str(exe)


@pytest.mark.parametrize("k", [0, 2, 3, 4])
def test_a_thread_that_cannot_start(program, k):
    # (allocation 1 is the list of the threads, one more for each of them)
    r = subprocess.run([program, str(k), "-1"], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "done 200\n"), r


@pytest.mark.parametrize("k,item", [(1, -1), (0, 0), (0, 199)])
def test_out_of_memory_before_the_threads_and_in_an_item(program, k, item):
    r = subprocess.run([program, str(k), str(item)], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout) == (0, "bad_alloc\n"), r
