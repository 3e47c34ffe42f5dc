"""Launches of more blocks than a dimension's threads allow (cube_nu_amd/csrc/grid.h):
every block has its place, and no dimension reaches 2^32 threads; or, in pieces, every
item has one, and no piece is larger than it may be.  The forms for few particles have
21 particles to a block of 64 threads, and take up to 2^32 - 257 particles (a recorded
call, or meshes of few tiles); in one launch they would end at 1.41e9.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cube_nu_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "grid.h"
int main() {
  const int64_t n[] = {1, 2, 63, (1 << 21) - 1, 1 << 21, (1 << 21) + 1, 1 << 23, 67108863, 67108864, 67974343,
                       (0xffffff00ll + 20) / 21};
  for (int64_t b : n) {
    const cube::Blocks g = cube::blocks_xy(b);
    const int64_t x = g.x, y = g.y;
    const bool ok = x > 0 && y > 0 && x * y >= b && x * (y - 1) < b && x * 1024 <= 0xffffffffll && y <= 65535 &&
                    (b > (1 << 21) || (y == 1 && x == b));
    if (!ok) { std::printf("%lld: %lld x %lld\n", (long long)b, (long long)x, (long long)y); return 1; }
  }
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_block_has_a_place(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout


PIECES = r"""
#include <cstdio>
#include "grid.h"
int main() {
  const int64_t cells = (int64_t)1 << 30, few = ((int64_t)1 << 25) * 21;
  const int64_t n[] = {1, 21, cells - 1, cells, cells + 1, 3ll * 1152 * 1152 * 1152, few, few + 1, 0xffffff00ll};
  for (int64_t most : {cells, few})
    for (int64_t k : n) {
      int64_t next = 0;
      bool ok = true;
      cube::in_pieces(k, most, [&](int64_t at, int64_t m) {
        ok = ok && at == next && m > 0 && m <= most;
        next = at + m;
      });
      if (!ok || next != k) { std::printf("%lld\n", (long long)k); return 1; }
    }
  std::puts(cells < 0xffffffffll && few / 21 * 64 < 0xffffffffll ? "ok" : "too large");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_pieces_hold_every_item_once(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PIECES)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
