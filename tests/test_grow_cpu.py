"""The ensemble's work lists (picard_amd/csrc/grow.h), compiled for the host: an allocation that fails, or
an old array that cannot be given up, leaves the array, its contents and its capacity as they were."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "grow.h"
int main() {
  int *p = nullptr, given = 0;
  int64_t cap = 0;
  bool full = false, stuck = false;
  auto alloc = [&](int **q, int64_t n) -> int {
    if (full) return -2;
    *q = (int *)std::calloc(n, sizeof(int));
    return 0;
  };
  auto give = [&](int *old) -> int {
    if (stuck) return -3;
    ++given;
    std::free(old);
    return 0;
  };
  auto grow = [&](int64_t want) { return picard::grow_array(&p, &cap, want, 3, alloc, give); };
  if (grow(10) || cap != 15 || !p) return 1;
  for (int i = 0; i < 45; ++i) p[i] = i;
  int *const was = p;
  if (grow(15) || p != was || given != 1) return 2;
  full = true;
  if (grow(16) != -2 || p != was || cap != 15 || given != 1) return 3;
  for (int i = 0; i < 45; ++i)
    if (p[i] != i) return 4;
  full = false;
  stuck = true;
  if (grow(16) != -3 || p != was || cap != 15) return 5;
  stuck = false;
  if (grow(16) || p == was || cap != 24 || given != 2) return 6;
  p[71] = 1;
  std::free(p);
  return 0;
}
"""


def test_a_failed_growth_changes_nothing(tmp_path):
    src = tmp_path / "grow.cpp"
    src.write_text(SRC)
    exe = tmp_path / "grow"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "picard_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.returncode
