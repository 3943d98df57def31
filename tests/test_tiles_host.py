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
