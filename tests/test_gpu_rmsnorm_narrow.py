"""Narrow rows (several per wave forward, up to 64 vectors backward): every lane count, row
counts around the workgroup's row slots and enough rows for several steps, against the oracle
with the suite's bars; the plan's coverage on the CPU."""
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

CSRC = Path(__file__).resolve().parent.parent / "trainscale_amd" / "csrc"
BF = torch.bfloat16

DRIVER = r"""
#include <cstdio>
#include <initializer_list>
#include "plan.hpp"
using namespace ts_plan;
static int fails = 0;
#define CHECK(c, ...) do { if (!(c)) { if (fails++ < 20) { std::printf(__VA_ARGS__); std::printf("\n"); } } } while (0)
int main() {
  for (long long nvec = 0; nvec <= 130; ++nvec) {
    const int f = rms_narrow_tpr(nvec);
    CHECK(f == 0 ? nvec == 0 || nvec > 32 : f >= nvec && (f == 8 || f == 16 || f == 32), "tpr");
    if (f != 0) CHECK(rms_fwd_plan(nvec).tpr == f && rms_fwd_plan(nvec).kv == 1, "forward lanes");
    for (long long rows : {1ll, 15ll, 16ll, 17ll, 127ll, 128ll, 129ll, 8192ll, 65537ll, 262144ll, 1ll << 30})
      for (int V : {4, 8}) {
        // what the launch takes: the plan of the size query and of the other sweeps
        const long long cols = nvec * V;
        const RmsBwdPlan p = rms_bwd_plan(rows, cols, 16 / V, true, true);
        CHECK(p.narrow == (nvec > 0 && nvec <= 64), "narrow");
        if (!p.narrow) continue;
        const RmsRowPlan& r = p.row;
        CHECK(r.tpr >= nvec && r.tpr <= 64 && r.kv == 1 && r.rpb * r.tpr == kNarrowBlock && !p.wave, "shape");
        CHECK(p.grid >= 1 && p.grid <= kBwdGridTarget && p.nparts == p.grid, "grid");
        CHECK(p.grid * p.steps * r.rpb >= rows, "rows not covered");
        CHECK((p.grid - 1) * p.steps * r.rpb < rows, "empty workgroup");
        CHECK(p.nparts <= rms_bwd_workspace_rows(rows, cols), "partial rows past the workspace");
        if (rows <= 129)
          for (long long wg = 0; wg < p.grid; ++wg)
            for (int sub = 0; sub < r.rpb; ++sub)
              for (long long st = 0; st < p.steps; ++st)
                for (int t = 0; t < r.tpr; ++t) {
                  const long long off = rms_bwd_load_offset(wg * r.rpb + sub, st, p.grid * r.rpb, p.steps,
                                                            rows, t, 0, r.tpr, V, nvec, cols);
                  CHECK(off >= 0 && off + V <= rows * cols, "load past the matrix");
                }
      }
  }
  std::printf("%d failures\n", fails);
  return fails != 0;
}
"""


def test_narrow_plan(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "n.cpp", tmp_path / "n"
    src.write_text(DRIVER)
    subprocess.run([gxx, "-O2", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    proc = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0, proc.stdout + proc.stderr


# columns: one vector, full and part-filled groups of 8, 16, 32 and 64 lanes; rows: one, around
# the row slots of a workgroup, and several steps of 512 workgroups
@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,dtype,wdtype", [
    (1, 8, BF, BF), (129, 64, BF, BF), (65, 72, BF, BF), (40000, 128, BF, BF),
    (63, 136, BF, torch.float32), (33, 256, BF, BF), (20001, 264, BF, BF), (17, 512, BF, BF),
    (70001, 64, torch.float16, torch.float16), (1000, 96, torch.float32, torch.float32),
    (31, 4, torch.float32, torch.float32), (9001, 256, torch.float32, torch.float32)])
def test_rows(gpu, rows, cols, dtype, wdtype):
    from test_gpu_rmsnorm import check_add, check_against_oracle
    g = torch.Generator(device=gpu).manual_seed(rows + cols)
    x, r, dy = ((torch.randn(rows, cols, generator=g, device=gpu)).to(dtype) for _ in range(3))
    w = (1 + 0.05 * torch.randn(cols, generator=g, device=gpu)).to(wdtype)
    check_against_oracle(x, w, dy, 1e-6)
    if rows <= 1000:
        check_add(x, r, w, dy, 1e-6)
