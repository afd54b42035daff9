"""The order of the atoms by distance (csrc/atom_order.h) on the CPU: sorted, and a
permutation also where coordinates are equal, infinite or not numbers (a place that no
atom takes would leave an index of the Becke force term unwritten)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_SOURCE = r"""
#include "atom_order.h"
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

int main() {
  std::mt19937 rng(5);
  const double odd[] = {NAN, -NAN, INFINITY, -INFINITY, 1e200, -1e200, 0.0, 5e-324};
  for (int n = 1; n <= 24; ++n)
    for (int rep = 0; rep < 40; ++rep) {
      std::vector<double> at(4 * n);
      for (double& v : at) v = (double)(int)(rng() % 7) - 3.0;  // many equal distances
      for (int k = 0; k < rep % 5; ++k) at[rng() % (4 * n)] = odd[rng() % 8];
      for (int a = 0; a < n; ++a) {
        std::vector<int> order(n, -1);
        for (int m = 0; m < n; ++m) {
          const int r = dg::distance_place(at.data(), n, a, m);
          if (r < 0 || r >= n || order[r] >= 0) return std::printf("n %d rep %d a %d m %d place %d\n", n, rep, a, m, r), 1;
          order[r] = m;
        }
        double last = 0.0;
        for (int m : order) {
          double d = 0.0;
          for (int k = 0; k < 3; ++k) d += (at[4 * m + k] - at[4 * a + k]) * (at[4 * m + k] - at[4 * a + k]);
          if (d < last) return std::printf("not sorted\n"), 1;
          if (d == d) last = d;
        }
      }
    }
  std::puts("order ok");
  return 0;
}
"""


def test_order_is_a_permutation(tmp_path):
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(_SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "dftcxx_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "order ok" in r.stdout, r.stdout
