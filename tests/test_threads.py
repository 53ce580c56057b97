"""Threads that a call can do without (csrc/host/threads.h), where the memory
for one of them is not to be had: the call goes on with those that it has, and
neither throws nor ends the process.  A small program of its own, whose
operator new fails at the n-th allocation."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dist_mem_gapbs_amd", "csrc")
PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include "host/threads.h"

static std::atomic<int> left{1 << 30};
void* operator new(std::size_t n) {
  if (left.fetch_sub(1) <= 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main(int, char** argv) {
  std::atomic<int> ran{0};
  std::thread helpers[3];
  int started = 0;
  left = std::atoi(argv[1]);
  for (auto& t : helpers) {
    if (!dmm::start_thread(&t, [&] { ran++; })) break;
    started++;
  }
  left = 1 << 30;
  for (auto& t : helpers)
    if (t.joinable()) t.join();
  std::printf("%d %d\n", started, ran.load());
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_no_memory_for_a_thread(tmp_path):
    src, exe = tmp_path / "t.cc", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    for allowed in range(4):  # one allocation a thread
        p = subprocess.run([str(exe), str(allowed)], capture_output=True, text=True)
        assert p.returncode == 0, (allowed, p.returncode, p.stderr)
        assert p.stdout.split() == [str(allowed), str(allowed)]
