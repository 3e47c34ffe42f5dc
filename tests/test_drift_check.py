"""The counts a drift compares (cube_nu_amd/csrc/drift_check.h), on the CPU: the ranked
particles with the placed ones in every drift, and with the physical particles where
the buffers are their images."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cube_nu_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "drift_check.h"
#define CHECK(c) do { if (!(c)) { std::printf("%s\n", #c); return 1; } } while (0)
int main() {
  using cube::drift_counts_agree;
  CHECK(drift_counts_agree(10, 10, true, 10));
  CHECK(drift_counts_agree(0, 0, true, 0));
  CHECK(!drift_counts_agree(9, 10, true, 10));    // a place without a particle
  CHECK(!drift_counts_agree(11, 10, false, -1));  // a particle without a place
  CHECK(!drift_counts_agree(9, 9, true, 10));     // lost with its source cell
  CHECK(!drift_counts_agree(11, 11, true, 10));   // taken twice
  CHECK(drift_counts_agree(9, 9, false, 10));     // buffers of their own
  CHECK(drift_counts_agree(9, 9, true, -1));      // physical particles not counted
  const long long big = 1ll << 33;
  CHECK(drift_counts_agree(big, big, true, big) && !drift_counts_agree(big, 0, false, -1));
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_counts_that_differ_are_found(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
