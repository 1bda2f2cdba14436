"""Columns and workgroup shapes of the cross-entropy kernels (ts_plan::tail_col,
ce_fused_plan), swept on the CPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "trainscale_amd" / "csrc"

DRIVER = r"""
#include <cstdio>
#include <initializer_list>
#include <vector>
#include "plan.hpp"
using namespace ts_plan;
static int fails = 0;
#define CHECK(c, ...) do { if (!(c)) { if (fails++ < 20) { std::printf(__VA_ARGS__); std::printf("\n"); } } } while (0)
int main() {
  for (int VE : {4, 8})
    for (long long V : {1, 2, 3, 5, 7, 8, 9, 15, 16, 17, 23, 24, 25, 1000, 50257}) {
      // every column once: whole vectors from column 0, then the lanes' tail elements
      std::vector<int> seen(V, 0);
      for (long long c = 0; c < V / VE * VE; ++c) seen[c]++;
      for (int t = 0; t < 1024; ++t) {
        const long long c = tail_col(V, t, VE);
        CHECK(c >= -1 && c < V, "tail column outside the row");
        if (c >= 0) seen[c]++;
      }
      for (long long c = 0; c < V; ++c) CHECK(seen[c] == 1, "column %lld of %lld held %d times", c, V, seen[c]);
    }
  // the shapes the launcher instantiates hold every row they are chosen for
  for (bool wide : {false, true})
    for (long long n = 0; n <= 20000; ++n) {
      const CeFusedPlan p = ce_fused_plan(n, wide);
      if (n > 16384) { CHECK(p.threads == 0, "too long"); continue; }
      CHECK((long long)p.threads * p.kv >= n, "row of %lld vectors does not fit", n);
      const bool known = (p.threads == 64 && p.kv == 4) || (p.threads == 256 && (p.kv == 4 || p.kv == 8 || p.kv == 16)) ||
                         (p.threads == 512 && p.kv == 16) || (p.threads == 1024 && p.kv == 16);
      CHECK(known && (!wide || p.threads == 1024), "no kernel for %d x %d", p.threads, p.kv);
    }
  std::printf("%d failures\n", fails);
  return fails != 0;
}
"""


def test_tail_columns_and_shapes(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "ce.cpp", tmp_path / "ce"
    src.write_text(DRIVER)
    subprocess.run([gxx, "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout + proc.stderr
