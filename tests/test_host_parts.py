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

POOL = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <thread>
#include "workspace.hpp"

// a device of g_cap bytes
static std::mutex g_m;
static std::map<void*, std::size_t> g_live;
static std::size_t g_used = 0, g_cap = 0;
static int g_allocs = 0;
static std::atomic<int> g_bad{0};
struct Dev {
  static bool alloc(void** p, std::size_t n) {
    std::lock_guard<std::mutex> g(g_m);
    ++g_allocs;
    if (g_used + n > g_cap) return false;
    *p = std::malloc(n);
    g_live[*p] = n;
    g_used += n;
    return true;
  }
  static void free(void* p) {
    std::lock_guard<std::mutex> g(g_m);
    auto it = g_live.find(p);
    if (it == g_live.end()) { ++g_bad; return; }
    g_used -= it->second;
    std::memset(p, 0xee, it->second);
    g_live.erase(it);
    std::free(p);
  }
};
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main() {
  {
    og::WorkspacePool<Dev> pool(400, 1000);
    og::Workspace a, b, c, d;
    g_cap = 1100;
    CHECK(pool.take(a, 300));
    void* p = a.p;
    pool.give(a);
    CHECK(pool.held() == 300 && pool.take(a, 200) && a.p == p && g_allocs == 1);  // kept and used again
    pool.give(a);
    CHECK(pool.take(a, 350) && g_used == 350);  // a larger one replaces it
    pool.give(a);
    CHECK(pool.take(b, 401));
    pool.give(b);
    CHECK(b.p == nullptr && g_used == 350);  // past the share of one owner
    CHECK(pool.take(b, 400) && pool.take(c, 300));
    pool.give(b);
    pool.give(c);
    CHECK(c.p == nullptr && pool.held() == 750 && g_used == 750);  // past the total
    // an allocation that fails takes the idle ones, not the one in use
    CHECK(pool.take(a, 100));
    void* q = nullptr;
    CHECK(pool.alloc(&q, 700) && b.p == nullptr && a.p != nullptr && pool.held() == 0);
    void* r = nullptr;
    CHECK(!pool.alloc(&r, 200));
    CHECK(!pool.take(d, 200) && d.p == nullptr && !d.busy);
    pool.give(a);
    CHECK(pool.take(d, 200) && a.p == nullptr);  // a's is idle now
    pool.drop(d);
    pool.drop(a);
    pool.drop(b);
    Dev::free(q);
    CHECK(g_used == 0 && pool.held() == 0 && g_live.empty());
  }
  // owners on four threads that fill what they use, on a device too small for all of them
  og::WorkspacePool<Dev> pool(600, 1500);
  g_cap = 2500;
  std::vector<std::thread> th;
  for (int t = 0; t < 4; ++t)
    th.emplace_back([&, t] {
      std::mt19937 rng(t);
      og::Workspace w[2];
      for (int i = 0; i < 20000; ++i) {
        og::Workspace& x = w[rng() & 1];
        const std::size_t n = 1 + rng() % 700;
        if (pool.take(x, n)) {
          std::memset(x.p, t, x.bytes);
          if (i % 7 == 0) std::this_thread::yield();
          for (std::size_t j = 0; j < x.bytes; ++j)
            if (static_cast<unsigned char*>(x.p)[j] != t) { ++g_bad; break; }
          pool.give(x);
        }
        if (i % 50 == 0) pool.drop(x);
      }
      pool.drop(w[0]);
      pool.drop(w[1]);
    });
  for (auto& x : th) x.join();
  CHECK(g_bad == 0 && g_used == 0 && pool.held() == 0 && g_live.empty());
  return 0;
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


def test_idle_workspaces_are_bounded_and_given_back(tmp_path):
    """What one owner and all owners keep is bounded, an allocation that fails takes the
    idle workspaces and none in use, and owners on several threads never lose theirs."""
    _run(tmp_path, "pool", POOL)
