"""The library's host-side parts that need no HIP, built for the host alone and driven by a
small program each."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STAGE = r"""
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>
#include "staging.hpp"

static bool g_fail = false;  // every operator new of the main thread throws
static thread_local bool t_main = false;
void* operator new(std::size_t n) {
  if (g_fail && t_main) throw std::bad_alloc();
  void* p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main() {
  t_main = true;
  for (int fail = 0; fail < 2; ++fail)
    for (std::size_t n : {std::size_t(1), std::size_t(3), std::size_t(7), std::size_t(1001)})
      for (int parts : {1, 4}) {
        std::vector<int> filled(n, 0), sent(n, 0);
        std::size_t next = 0;
        int waits = 0;
        g_fail = fail;
        const int rc = og::stage(
            n, parts, [&](std::size_t a, std::size_t b) { for (; a < b; ++a) ++filled[a]; },
            [&](std::size_t a, std::size_t b) {
              if (a != next) return 7;
              for (next = b; a < b; ++a) sent[a] += filled[a];
              return 0;
            },
            [&] { ++waits; return 0; });
        g_fail = false;
        if (rc != 0 || next != n || waits != 1) return std::printf("rc %d, %zu of %zu\n", rc, next, n), 1;
        for (std::size_t i = 0; i < n; ++i)
          if (filled[i] != 1 || sent[i] != 1) return std::printf("element %zu of %zu\n", i, n), 1;
      }
  // an error ends the sending, not the filling, and what was sent is waited for
  std::vector<int> filled(8, 0);
  int sends = 0, waits = 0;
  const int rc = og::stage(
      8, 4, [&](std::size_t a, std::size_t b) { for (; a < b; ++a) ++filled[a]; },
      [&](std::size_t, std::size_t) { return ++sends == 2 ? 5 : 0; }, [&] { ++waits; return 6; });
  for (int f : filled)
    if (f != 1) return 1;
  return rc == 5 && sends == 2 && waits == 1 ? 0 : 1;
}
"""


def _run(tmp_path, name, source):
    cxx = shutil.which("g++") or shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
    if not os.path.exists(cxx):
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / f"{name}.cpp", tmp_path / name
    src.write_text(source)
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "ocean_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)


def test_staging_fills_every_part_without_threads_or_memory(tmp_path):
    """Parts filled once and sent in order, with threads and where none can be had (the
    allocation of a thread's state fails): no exception passes a C entry point."""
    _run(tmp_path, "stage", STAGE)
