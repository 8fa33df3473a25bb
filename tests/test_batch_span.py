"""Substeps planned ahead of their launches (mpm_amd/csrc/span.hpp) under
errors, on the CPU: whichever step fails, the bookkeeping ends where the
launches do, and the substeps planned before a planning error still run."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CXX = shutil.which("g++")

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include "span.hpp"

struct Ops {
  int n, plan_fails, launch_fails, begin_fails, end_fails, cycle;
  int host = 0, device = 0, begun = 0, ended = 0;  // substeps on the books, substeps launched
  int save() const { return host; }
  void restore(int h) { host = h; }
  int plan(int i) {
    if (i == plan_fails) { host += 1000; return 1; }  // (partly planned)
    ++host;
    return 0;
  }
  bool more(int planned) { return planned != cycle; }
  int begin() { ++begun; return begin_fails ? 2 : 0; }
  int launch(int i) { if (i == launch_fails) return 3; ++device; return 0; }
  int end() { ++ended; return end_fails ? 4 : 0; }
};

#define CHECK(c) if (!(c)) { std::printf("%s: n %d plan %d launch %d begin %d end %d cycle %d: host %d device %d ran %d rc %d\n", \
    #c, n, p, l, b, e, cycle, o.host, o.device, ran, rc); return 1; }

int main() {
  int cases = 0;
  for (int n = 1; n <= 4; ++n)
    for (int p = -1; p <= n; ++p)
      for (int l = -1; l <= n; ++l)
        for (int b = 0; b < 2; ++b)
          for (int e = 0; e < 2; ++e)
            for (int cycle = 1; cycle <= 5; ++cycle) {
              Ops o{n, p, l, b, e, cycle};
              int ran = -1;
              const int rc = mpm_engine::run_span(o, n, &ran);
              const int last = n < cycle ? n : cycle;
              const bool bad_plan = p >= 0 && p < last;
              const int planned = bad_plan ? p : last;
              const int want = planned == 0 || b ? 0 : l >= 0 && l < planned ? l : planned;
              CHECK(o.host == o.device)
              CHECK(o.device == want && ran == want)
              CHECK(o.begun == (planned > 0) && o.ended == 1)
              CHECK(rc == (planned > 0 && b ? 2 : planned > 0 && l >= 0 && l < planned ? 3 : bad_plan ? 1 : e ? 4 : 0))
              ++cases;
            }
  std::printf("%d cases\n", cases);
  return 0;
}
"""


@pytest.mark.skipif(CXX is None, reason="no g++")
def test_books_and_launches_agree_after_any_error(tmp_path):
    src, exe = tmp_path / "span.cpp", tmp_path / "span"
    src.write_text(DRIVER)
    subprocess.run([CXX, "-std=c++17", "-O1", "-Wall", "-Wextra", "-I", str(ROOT / "mpm_amd" / "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
    assert int(out.stdout.split()[0]) > 1000
