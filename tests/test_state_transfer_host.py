"""The host side of a state transfer's chunks (no GPU): every chunk is done once
and nothing is thrown, also where no helper thread can be started.

A small program is built around the header, with an operator new that fails from a
given allocation on: starting a thread allocates."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sphpc_amd",
                    "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include "sph_io.h"
static std::atomic<long> left{1L << 40};
void *operator new(std::size_t n) {
  if (left.fetch_sub(1) <= 0) throw std::bad_alloc();
  if (void *p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, std::size_t) noexcept { std::free(p); }
extern "C" int transfer(size_t chunks) {  // as a C entry: nothing may be thrown
  static std::atomic<int> done[64];
  for (auto &d : done) d = 0;
  int calls = 0;
  sph::io_chunks(chunks, sph::kIoThreads, [&](size_t k) { done[k]++; }, [&]() { ++calls; });
  for (size_t k = 0; k < 64; ++k)
    if (done[k] != (k < chunks ? 1 : 0)) return 1;
  return calls > 0 ? 0 : 1;
}
int main() {
  for (long allowed = 0; allowed < 12; ++allowed)
    for (size_t chunks : {0, 1, 2, 3, 16, 64}) {
      left = allowed;
      const int bad = transfer(chunks);
      left = 1L << 40;
      if (bad) return 1;
    }
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_chunks_without_memory_for_threads(tmp_path):
    src, exe = tmp_path / "io.cc", tmp_path / "io"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True, timeout=100)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stderr)
