"""The pinned blocks that downloads share (mpm_amd/csrc/slot_pool.hpp), on the
CPU with ordinary memory: how many there are, that they are used again and given
back, that no two calls hold one block, that nobody waits."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CXX = shutil.which("g++")

DRIVER = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include "slot_pool.hpp"

std::atomic<int> live{0}, made{0};
bool none_left = false;
struct Memory {
  static uint8_t* make(size_t bytes) {
    if (none_left) return nullptr;
    ++live; ++made;
    return (uint8_t*)std::malloc(bytes);
  }
  static void drop(uint8_t* p) { --live; std::free(p); }
};
using Pool = mpm_engine::SlotPool<Memory, 4, 32>;
#define CHECK(c) if (!(c)) { std::printf("line %d: %s (live %d, made %d)\n", __LINE__, #c, (int)live, (int)made); std::exit(1); }

int main() {
  Pool pool;
  Pool::Slot a[8], b[8], c[8];
  pool.attach();
  pool.attach();
  CHECK(pool.take(1, 100, a) == 1 && live == 1);
  std::memset(a[0].p, 1, 100);
  pool.give(a, 1);
  CHECK(pool.take(1, 60, b) == 1 && b[0].p == a[0].p && made == 1);  // used again
  pool.give(b, 1);
  CHECK(pool.take(3, 1000, a) == 3 && live == 4);   // beside the small one
  CHECK(pool.take(2, 1000, b) == 1 && live == 4);   // the small one makes way
  CHECK(pool.take(8, 1000, c) == 1 && live == 5);   // none left: one for this call
  pool.give(c, 1);
  CHECK(live == 4);
  pool.give(a, 3);
  pool.give(b, 1);
  CHECK(live == 4 && pool.take(8, 10, a) == 4 && live == 4);
  pool.give(a, 4);
  pool.detach();
  CHECK(live == 4);
  pool.detach();
  CHECK(live == 0);                                 // the last user gives all back
  made = 0;
  pool.attach();
  for (size_t bytes = 1000; bytes < 1064; ++bytes) {  // a call that grows: one block for every 32 bytes more
    CHECK(pool.take(1, bytes, a) == 1 && a[0].bytes >= bytes);
    pool.give(a, 1);
  }
  CHECK(made == 3 && live == 3);
  pool.detach();
  none_left = true;
  CHECK(pool.take(2, 10, a) == 0);
  none_left = false;
  // many threads: a block is in one pair of hands
  std::atomic<int> torn{0};
  auto work = [&](int id) {
    pool.attach();
    for (int i = 0; i < 2000; ++i) {
      Pool::Slot s[3];
      const size_t bytes = 64 + 64 * (size_t)((id + i) % 3), n = pool.take(1 + (size_t)(i % 3), bytes, s);
      if (n == 0) ++torn;
      for (size_t k = 0; k < n; ++k) std::memset(s[k].p, id, bytes);
      for (size_t k = 0; k < n; ++k)
        for (size_t q = 0; q < bytes; ++q) torn += s[k].p[q] != (uint8_t)id;
      if (live > 4 + 8) ++torn;
      pool.give(s, n);
    }
    pool.detach();
  };
  std::thread t[8];
  for (int i = 0; i < 8; ++i) t[i] = std::thread(work, i + 1);
  for (auto& x : t) x.join();
  CHECK(torn == 0 && live == 0);
  std::printf("ok\n");
  return 0;
}
"""


@pytest.mark.skipif(CXX is None, reason="no g++")
def test_blocks_are_shared_bounded_and_given_back(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(DRIVER)
    subprocess.run([CXX, "-std=c++17", "-O1", "-Wall", "-Wextra", "-pthread", "-I", str(ROOT / "mpm_amd" / "csrc"),
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "ok\n", out.stdout
