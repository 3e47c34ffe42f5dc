"""The kick's meshes within the workspace budget (cube_nu_amd/csrc/plan.h), on the CPU:
under a budget that the caller has set, the tile meshes held at once and the
whole-image mesh together stay within it wherever one mesh of the largest level
does; the automatic budget is that of the tile meshes."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cube_nu_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "plan.h"
using namespace cube;
#define CHECK(c) do { if (!(c)) { std::printf("%s at ng %lld, budget %lld\n", #c, (long long)ng, (long long)budget); return 1; } } while (0)
int main() {
  long taken = 0, batches = 0;
  for (int64_t ng : {16, 48, 64, 96, 128, 192, 320, 448, 512, 1024}) {
    const int64_t nnt = ng % 64 ? 2 : 4, tile = ng / nnt + 32, sub = 2 * (ng / nnt / 2) + 16;  // meshes of the levels
    const int64_t sizes[] = {ng / 4, tile, sub, 2 * sub}, image = 4 * 8 * ng * ng * ng;
    int64_t largest = 0;
    for (int64_t n : sizes) largest = std::max(largest, mesh_bytes(n, 4) + face_bytes(n));
    for (int64_t budget = 1; budget < ((int64_t)1 << 38); budget += budget / 3 + 1) {
      for (bool set : {false, true}) {
        const bool fits = image_fits(budget, set, image, largest);
        CHECK(!fits || 2 * image <= budget);
        const int64_t reserved = fits ? image : 0;
        for (int64_t n : sizes)
          for (bool faces : {false, true}) {
            if (faces && !fits) continue;
            const int64_t per = mesh_bytes(n, 4) + (faces ? face_bytes(n) : 0);
            for (int64_t nmesh : {1, 64, 4096}) {
              const int64_t b = level_batch(budget, set, reserved, per, nmesh);
              CHECK(b >= 1 && b <= nmesh);
              CHECK(b == 1 || b * per + (set ? reserved : 0) <= budget);
              if (set && largest + reserved <= budget) CHECK(b * per + reserved <= budget);
              CHECK(b == nmesh || (b + 1) * per + (set ? reserved : 0) > budget);
              taken += fits;
              batches += fits && b < nmesh;
            }
          }
      }
    }
  }
  std::printf(taken > 1000 && batches > 100 ? "ok\n" : "few\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_meshes_stay_within_the_budget(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
