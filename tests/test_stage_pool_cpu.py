"""The pool of staging buffers (csrc/stage_pool.h): bounded, the smallest buffer that fits, and calls with larger
tables keep theirs after a batch of small ones has filled it.  Compiled and run on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "stage_pool.h"
using fmm2d::StagePool;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
static char mem[64];
int main() {
  const size_t K = 1024, M = K * K;
  StagePool P;
  CHECK(P.take(1).p == nullptr);
  // a batch of small calls on 8 streams (and of 16) leaves its buffers ...
  for (int k = 0; k < 16; ++k) CHECK(P.give({mem + k, (256 + 16 * k) * K}).empty());
  // ... then calls with 3 MiB of tables: the first allocates, the others find its buffer
  CHECK(P.take(3 * M).p == nullptr);
  const auto gone = P.give({mem + 20, 3 * M});
  CHECK(gone.size() == 1 && gone[0].p == mem);  // the oldest
  for (int k = 0; k < 3; ++k) {
    const auto b = P.take(3 * M);
    CHECK(b.p == mem + 20 && b.cap == 3 * M);
    CHECK(P.give(b).empty());
  }
  // the smallest that fits
  const auto s = P.take(300 * K);
  CHECK(s.p == mem + 3 && s.cap == 304 * K);
  // bytes are bounded too, and a buffer beyond the bound is not kept
  CHECK(!P.give({mem + 21, StagePool::kBytes}).empty() && P.free.size() == 1 && P.free[0].p == mem + 21);
  const auto all = P.give({mem + 22, StagePool::kBytes + 1});
  CHECK(all.size() == 2 && all[1].p == mem + 22 && P.free.empty());
  // large and small in turn: both stay
  P.give({mem + 30, 8 * M});
  for (int k = 0; k < 8; ++k) P.give({mem + 31 + k, 256 * K});
  for (int k = 0; k < 50; ++k) {
    const auto a = P.take(8 * M), b = P.take(100 * K);
    CHECK(a.p == mem + 30 && b.p && b.cap == 256 * K);
    CHECK(P.give(b).empty() && P.give(a).empty());
  }
  return 0;
}
"""


def test_pool_rule(tmp_path):
    src, exe = tmp_path / "pool.cpp", tmp_path / "pool"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "fmm2d_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
