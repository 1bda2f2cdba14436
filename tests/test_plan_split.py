"""K split of the linear-CE's grad_hidden GEMM (ts_plan::hidden_split, gemm_piece_of), swept
on the CPU: the pieces are a bijection onto (slot, M-tile, N-tile), the slots' K ranges cover
K exactly and start on a k-block, and the byte counts the workspace queries report cover the
partials of every shape."""
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
  for (long long MT : {1, 2, 5, 16, 33})
    for (long long NT : {1, 3, 16})
      for (long long S : {1, 2, 5, 21}) {
        std::vector<char> seen(MT * NT * S, 0);
        for (long long b = 0; b < MT * NT * S; ++b) {
          int64_t s, mt, nt;
          gemm_piece_of(b, MT, NT, S, s, mt, nt);
          const bool ok = s >= 0 && s < S && mt >= 0 && mt < MT && nt >= 0 && nt < NT;
          CHECK(ok, "piece %lld of %lld x %lld x %lld", b, MT, NT, S);
          if (!ok) continue;
          CHECK(!seen[(s * MT + mt) * NT + nt], "piece visited twice");
          seen[(s * MT + mt) * NT + nt] = 1;
        }
      }
  for (long long M : {1, 8, 255, 256, 257, 1000, 2048, 4096, 32768, 40000})
    for (long long H : {8, 64, 256, 264, 768, 4096, 16384})
      for (long long K : {1, 31, 32, 4095, 4096, 4097, 8192, 16390 * 32, 50257, 128256, 1 << 22}) {
        const KSplit k = hidden_split(M, H, K);
        CHECK(k.splits >= 1 && k.kper % kGemmBlockK == 0 && k.kper > 0, "split");
        CHECK(k.splits * k.kper >= K, "slots do not cover K");
        const long long tiles = ((M + 255) / 256) * ((H + 255) / 256);
        CHECK(k.splits == 1 || k.splits * tiles <= kCus, "more pieces than CUs");
        CHECK(k.splits == 1 || k.kper >= kSplitMinBlocks * kGemmBlockK, "short slots");
        const long long bytes = hidden_split_bytes(M, H, K);
        CHECK(bytes == (k.splits > 1 ? k.splits * M * H * 4 : 0), "bytes");
        CHECK(bytes <= hidden_split_bytes_any_h(M, K), "bound without H (%lld %lld %lld)", M, H, K);
        CHECK(bytes <= hidden_split_bytes_any_shape(M), "bound without H and K");
        // a shorter last chunk of the same split: slots cover it, some may be empty
        for (long long last : {1ll, K / 3 + 1, K})
          CHECK(k.splits * split_kper(last, k.splits) >= last, "last chunk");
      }
  // the bound is met by some H, and a few rows do not ask for what a full tile of them would
  for (long long M : {1, 8, 256, 300, 2048, 32768}) {
    long long most = 0;
    for (long long ht = 1; ht <= 256; ++ht) {
      const long long b = hidden_split_bytes(M, ht * 256, 1ll << 40);
      most = b > most ? b : most;
    }
    CHECK(most == hidden_split_bytes_any_shape(M), "bound of %lld rows: %lld, needed %lld", M,
          (long long)hidden_split_bytes_any_shape(M), most);
  }
  // a tile for every CU: one slot
  CHECK(hidden_split(4096, 4096, 128256).splits == 1, "C5 chunk is not split");
  CHECK(hidden_split(1024, 768, 50257).splits == 21, "12 tiles");
  std::printf("%d failures\n", fails);
  return fails != 0;
}
"""


def test_hidden_split(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "split.cpp", tmp_path / "split"
    src.write_text(DRIVER)
    subprocess.run([gxx, "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout + proc.stderr
