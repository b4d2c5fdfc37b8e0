"""The host thread pool (ccq_amd/csrc/pool.h) on the CPU: every chunk is taken
once, also when an allocation for the pool or one of its threads fails."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include "pool.h"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
static std::atomic<int> left{-1};   // allocations until one fails
void* operator new(std::size_t n) {
  if (left >= 0 && left-- == 0) throw std::bad_alloc();
  void* p = std::malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
int main(int, char** argv) {
  std::atomic<int> next{0}, done{0};
  left = std::atoi(argv[1]);
  ccqpool::run(std::atoi(argv[2]), [&](int) {
    while (next++ < 1000) ++done;
  });
  left = -1;
  std::printf("%d\n", done.load());
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "t.cpp").write_text(SRC)
    exe = str(d / "t")
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-pthread", "-I",
                    os.path.join(ROOT, "ccq_amd", "csrc"), str(d / "t.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("fail", [-1, 0, 1, 2, 5])
@pytest.mark.parametrize("n", [1, 2, 8])
def test_pool_finishes_the_job(program, fail, n):
    r = subprocess.run([program, str(fail), str(n)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stderr)
    assert r.stdout.strip() == "1000"
