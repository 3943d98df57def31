"""plan_tile (csrc/gk_fp8_plan.h): the GPU tests' shapes reach every tile, and a full chip keeps 256 x 256 tiles."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "gaudi-kernels_amd" / "csrc"
SRC = """#include <cstdio>
#include "gk_fp8_plan.h"
int main() { int m, n; while (std::scanf("%d %d", &m, &n) == 2)
  std::printf("%d\\n", gk::plan_tile(m, (m + 255) / 256 * 256, n, 256)); }
"""


def test_plan_tile(tmp_path):
    exe = tmp_path / "plan_tile"
    (tmp_path / "p.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(tmp_path / "p.cpp"), "-o", str(exe)], check=True)
    shapes = [(65, 500), (128, 6140), (300, 6144), (777, 5003), (1000, 4090), (4096, 6144), (4096, 7168),
              (1024, 28672)]
    out = subprocess.run([str(exe)], input="\n".join(f"{m} {n}" for m, n in shapes), check=True, capture_output=True,
                         text=True).stdout.split()
    assert [int(v) for v in out] == [0, 1, 2, 3, 4, 5, 5, 5]

FORM_SRC = """#include <cstdio>
#include "gk_fp8_plan.h"
int main() { int m, n, k, form, wide; while (std::scanf("%d %d %d %d %d", &m, &n, &k, &form, &wide) == 5)
  std::printf("%d\\n", gk::plan_tile(m, (m + 255) / 256 * 256, n, 256, k / 128, gk::TileForm(form), wide, wide)); }
"""
OCP, HALF, CHANNEL = 0, 1, 2
# (m, n, k, form, wide output rows) -> tile: 64x32, 64x64, 128x64, 128x64 twice a CU, 128x128, 256x256
FORM_CASES = [
    # half range converts each wave's weight fragments: 256 x 256 tiles (8 token blocks a fragment) take over earlier
    ((700, 6144, 14336, HALF, 1), 5), ((1400, 4096, 14336, HALF, 1), 5), ((2617, 5923, 6400, HALF, 0), 5),
    ((4096, 2048, 2048, HALF, 1), 5), ((300, 6144, 4096, HALF, 1), 2), ((1024, 4096, 4096, HALF, 1), 4),
    # two full rounds of 128 x 128 tiles lose to 128 x 64 tiles, or to 256 x 256 ones on half the CUs
    ((4096, 2048, 2048, OCP, 1), 3), ((8192, 1024, 512, CHANNEL, 1), 5), ((512, 14336, 512, CHANNEL, 1), 5),
    # rows without wide stores cost the 256 x 256 tile most
    ((600, 23990, 256, HALF, 0), 4), ((600, 23990, 256, HALF, 1), 5),
    # the shapes of the GPU tests: every tile in every form
    ((65, 500, 384, OCP, 1), 0), ((128, 6140, 640, OCP, 1), 1), ((300, 6144, 640, OCP, 1), 2),
    ((777, 5003, 384, OCP, 0), 3), ((1000, 4090, 896, OCP, 1), 4), ((4096, 6144, 256, OCP, 1), 5),
    ((4096, 6144, 8320, OCP, 1), 5), ((4096, 6144, 384, OCP, 1), 5), ((4096, 6144, 128, OCP, 1), 5),
    *(((m, n, k, form, wide), 5) for m, n in ((2040, 7163), (3000, 6001)) for k in (1152, 256, 384, 512)
      for form in (OCP, HALF) for wide in (0, 1)),  # test_gpu_prefill256.py
    ((65, 500, 384, HALF, 1), 0), ((128, 6140, 640, HALF, 1), 1), ((300, 6144, 640, HALF, 1), 2),
    ((777, 5003, 384, HALF, 0), 3), ((1000, 4090, 896, HALF, 1), 4),
    ((17, 500, 384, CHANNEL, 1), 0), ((128, 6140, 640, CHANNEL, 1), 1), ((300, 6144, 256, CHANNEL, 1), 2),
    ((777, 5003, 384, CHANNEL, 0), 3), ((640, 4090, 2048, CHANNEL, 1), 4), ((2047, 7168, 256, CHANNEL, 1), 5),
]


def test_plan_tile_forms(tmp_path):
    exe = tmp_path / "plan_tile"
    (tmp_path / "p.cpp").write_text(FORM_SRC)
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(tmp_path / "p.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c, _ in FORM_CASES), check=True,
                         capture_output=True, text=True).stdout.split()
    assert [(c, int(v)) for (c, _), v in zip(FORM_CASES, out)] == FORM_CASES


def test_column_ranges(tmp_path):
    """test_gpu_prefill256.py: one column range of 256-wide tiles, and two."""
    (tmp_path / "p.cpp").write_text("""#include "gk_fp8_plan.h"
int main() { return gk::prefill_wide_columns(2048, 7163, 256) == 7163 && gk::prefill_wide_columns(3072, 6001, 256) == 2048 ? 0 : 1; }
""")
    exe = tmp_path / "p"
    subprocess.run(["g++", "-std=c++17", "-I", str(CSRC), str(tmp_path / "p.cpp"), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
