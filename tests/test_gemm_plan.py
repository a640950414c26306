"""The choice of the GEMM kernels (csrc/gemm_plan.hpp), checked on the CPU.

For a wide range of routed rows, expert counts and widths: the choice is one
the kernels have, the tile table's bound holds the tiles of every choice at
any row count up to the bound's, and padded widths never split K over waves
(so that their results do not depend on the row count).  At sizes where one
kernel measured far ahead of the other the choice is that one.
"""
import os
import shutil
import subprocess

import pytest

from gemm_cases import DENSE, EXPERTS, ONE_EXPERT

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
           // routed; dense without and with a copy of x to save; a shared branch with half of the rows
           for (double copy : {-1.0, 0.0, 20.0, -2.0}) {
            if (copy >= 0 && E != 1) continue;
            const GemmPlan p = gemm_plan(dt, A, E, Dk, Hp, D, H, copy, copy == -2.0 ? A / 2 : 0);
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


# (dtype, routed rows, experts, dim, hidden, GEMM, tile rows): stage times on one
# MI355X in us, 256-row tiles against the best of gemm_rows
MEASURED = [
    ("bf16", 5539, 1, 512, 768, "up", 256),        # 20.0 against 38.7
    ("bf16", 2836, 1, 512, 1408, "up", 256),       # 20.1 against 36.6
    ("bf16", 2567, 1, 768, 1536, "up", 256),       # 24.4 against 43.3
    ("bf16", 19116, 4, 256, 256, "up", 256),       # 16.5 against 30.3
    ("bf16", 16000, 32, 256, 640, "up", 256),      # a forward 76 against 104
    ("bf16", 4000, 32, 512, 2048, "up", 256),      # 42.3 against 68.1
    ("f32", 7322, 16, 1024, 1024, "up", 256),      # 161 against 259
    ("bf16", 14560, 64, 616, 616, "down", 256),    # 27.7 against 45.5
    ("bf16", 15361, 64, 1216, 304, "up", 256),     # 48.9 against 76.3
    ("bf16", 32, 8, 1536, 4096, "up", 16),         # 37 against 28
    ("bf16", 2222, 6, 1000, 2667, "down", 64),     # 53 against 35
    ("f32", 416, 4, 64, 128, "up", 16),            # a forward 59 against 31
]

PICKS = r"""
#include "gemm_plan.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
using namespace nomas;
int main(int argc, char** argv) {
  for (int i = 1; i + 5 < argc; i += 6) {
    const DType dt = !strcmp(argv[i], "f32") ? DType::F32 : !strcmp(argv[i], "bf16") ? DType::BF16 : DType::F16;
    const int64_t A = atol(argv[i + 1]), E = atol(argv[i + 2]), D = atol(argv[i + 3]), H = atol(argv[i + 4]);
    const int64_t Dk = padded_k(D, (int)dtype_size(dt)), Hp = round_up(H, 128), mt = (A + 255) / 256;
    const GemmPlan p = gemm_plan(dt, A, E, Dk, Hp, D, H, atof(argv[i + 5]));
    // the K-split parts of one expert's last tiles (tile_map.hpp)
    const int turn = kStages * kKBlockBytes / (int)dtype_size(dt);
    const bool padded = D % 256 || H != Hp;
    const int s1 = padded ? 1 : split_parts(mt * (2 * Hp / 256), (int)(Dk / turn));
    const int s2 = padded ? 1 : split_parts(mt * (round_up(D, 256) / 256), (int)(Hp / turn));
    printf("%d %d %d %d %d %d\n", p.bm1, p.waves1, p.bm2, p.waves2, s1, s2);
  }
  return 0;
}
"""


def picks(tmp_path, calls):
    """(bm1, waves1, bm2, waves2, parts1, parts2) of each (dtype, routed rows, experts, dim,
    hidden, dense_copy); the parts are those of one expert."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    src = tmp_path / "picks.cpp"
    src.write_text(PICKS)
    exe = tmp_path / "picks"
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-I", CSRC,
                    str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)] + [str(v) for c in calls for v in c], capture_output=True,
                         text=True, timeout=60, check=True).stdout.split("\n")
    return [tuple(int(v) for v in line.split()) for line in out if line]


def test_measured_choices(tmp_path):
    got = picks(tmp_path, [c[:5] + (-1,) for c in MEASURED])
    for c, p in zip(MEASURED, got):
        assert (p[0] if c[5] == "up" else p[2]) == c[6], (c, p)


def test_calls_reach_gemm_mfma(tmp_path):
    """The calls of gemm_cases.py run the 256-row kernel in the forms they name."""
    one = [(dt, rows, 1, D, H, copy) for cases, copy in ((ONE_EXPERT, -1), (DENSE, 0))
           for dt, rows, D, H, _, _ in cases]
    want = [c[4:] for c in ONE_EXPERT + DENSE]
    for call, parts, p in zip(one, want, picks(tmp_path, one)):
        assert p[0] == 256 and p[2] == 256 and p[4:] == parts, (call, p)
    several = [(dt, rows * k, E, D, H, -1) for dt, rows, D, E, k, H in EXPERTS]
    for call, p in zip(several, picks(tmp_path, several)):
        assert p[0] == 256 and p[2] == 256, (call, p)
