"""The deposit's bisection (picard_amd/csrc/bisect.h) at positions whose sum is beyond
2^31, compiled for the host: a sequence that is its own formula stands in for the array."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <initializer_list>
#include "bisect.h"
struct Descending {
  int lo, hi;                            // what may be read
  mutable bool bad = false;
  int32_t operator[](int i) const {
    if (i < lo || i >= hi) { bad = true; return 0; }
    return 2147483647 - i;
  }
};
int main() {
  const int starts[] = {0, 1000, (1 << 30) - 60, 1 << 30, 1074262985, 2147483647 - 400};
  for (int lo : starts)
    for (int n : {0, 1, 2, 3, 127, 128, 200})
      for (int take = 0; take <= n; ++take) {
        Descending d{lo, lo + n};
        const int32_t q = 2147483647 - (lo + take);          // `take` entries are greater
        const int got = picard::greater_in(d, lo, lo + n, q);
        if (got != take || d.bad) { std::printf("lo %d n %d: %d of %d\n", lo, n, got, take); return 1; }
      }
  return 0;
}
"""


def test_bisection_beyond_2_31(tmp_path):
    src = tmp_path / "bisect.cpp"
    src.write_text(SRC)
    exe = tmp_path / "bisect"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "picard_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
