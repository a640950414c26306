"""The choice of the GEMM kernels (csrc/gemm_plan.hpp), checked on the CPU.

For a wide range of routed rows, expert counts and widths: the choice is one
the kernels have, the tile table's bound holds the tiles of every choice at
any row count up to the bound's, and padded widths never split K over waves
(so that their results do not depend on the row count).
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "hy-nomas-rs_amd", "csrc")

PROG = r"""
#include "gemm_plan.hpp"
#include <cstdio>
using namespace nomas;
int main() {
  long n = 0, mixed = 0, used[4] = {0, 0, 0, 0};
  const int64_t widths[] = {8, 64, 72, 256, 264, 1000, 1024, 1536, 3072};
  const int64_t hiddens[] = {1, 96, 128, 640, 2667, 4096, 8192};
  for (DType dt : {DType::F32, DType::BF16, DType::F16})
    for (int64_t E : {1, 2, 7, 8, 17, 64, 257})
      for (int64_t D : widths)
        for (int64_t H : hiddens) {
          const int64_t Dk = padded_k(D, (int)dtype_size(dt)), Hp = round_up(H, 128);
          int64_t most = 0;  // tiles of any call so far (A ascending)
          for (int64_t A = 1; A < 40000000; A += 1 + A / 7) {
            const GemmPlan p = gemm_plan(dt, A, E, Dk, Hp, D, H);
            const int bms[2] = {p.bm1, p.bm2}, waves[2] = {p.waves1, p.waves2};
            for (int g = 0; g < 2; ++g) {
              const int bm = bms[g];
              const bool rows = bm == 16 || bm == 32 || bm == 64;
              if (!rows && bm != kMfmaBM) { printf("tile of %d rows\n", bm); return 1; }
              if (rows != (waves[g] > 0)) { printf("waves\n"); return 1; }
              if (rows && (D % 256 || H % 128) && waves[g] != 1) { printf("order\n"); return 1; }
              const int64_t tiles = (A + bm - 1) / bm + E;
              most = tiles > most ? tiles : most;
              if (most > max_gemm_tiles(A, E)) { printf("bound: A %ld E %ld\n", (long)A, (long)E); return 1; }
              used[bm == 16 ? 0 : bm == 32 ? 1 : bm == 64 ? 2 : 3]++;
            }
            mixed += p.bm1 != p.bm2;
            ++n;
          }
        }
  if (!mixed) { printf("the GEMMs never differ\n"); return 1; }
  for (long u : used) if (!u) { printf("a choice is never taken\n"); return 1; }
  printf("ok %ld\n", n);
  return 0;
}
"""


def test_gemm_plan(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src = tmp_path / "gemm_plan_check.cpp"
    src.write_text(PROG)
    exe = tmp_path / "gemm_plan_check"
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-I", CSRC,
                    str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.startswith("ok")
