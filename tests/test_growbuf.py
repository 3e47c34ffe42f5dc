"""Arrays a captured call has used stay allocated when a later call needs larger ones
(cube_nu_amd/csrc/growbuf.h), on the CPU with a counting allocator: a graph
replayed after such a growth would otherwise read and write freed memory.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cube_nu_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "growbuf.h"
static std::map<void*, int> frees;
static bool none = false;
struct Mem {
  static void* alloc(std::size_t b) { if (none) throw 1; void* p = std::malloc(b); frees[p] = 0; return p; }
  static void free(void* p) { ++frees[p]; }  // (addresses are never reused)
};
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
  void *a, *b, *c, *d;
  {
    cube::GrowBuf<int, Mem> q;
    q.hold();                                    // of nothing
    a = q.ensure(4);
    CHECK(q.ensure(3) == a && q.n == 4);
    b = q.ensure(8);                             // no capture has seen a
    CHECK(a != b && frees[a] == 1);
    q.hold();                                    // a capture sees b
    CHECK(q.ensure(8) == b);
    c = q.ensure(16);
    CHECK(c != b && frees[b] == 0);              // the graph still holds b
    d = q.ensure(32);
    CHECK(frees[c] == 1 && frees[b] == 0);       // none has seen c
    q.hold();
    none = true;
    bool threw = false;
    try { q.ensure(64); } catch (int) { threw = true; }
    CHECK(threw && q.p == nullptr && q.n == 0 && frees[d] == 0);
    none = false;
    CHECK(q.ensure(64) != nullptr);
  }
  for (auto& f : frees) CHECK(f.second == 1);    // each freed once in the end
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_arrays_of_captured_calls_outlive_growth(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
