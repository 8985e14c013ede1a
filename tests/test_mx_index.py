"""Plane indices of the matrix-core B kernel on the CPU: every plane that a
wavefront requests (the ring's and the one ahead, from any first cell) lies in
the grid, for the windows and the shortest first axes that the fast path
takes (n0 = 2m + 3 up).  And the ragged bins cover their axis."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "mx_index.hpp"
using namespace nfft_hip;
int main() {
  int bad = 0;
  for (int m = 1; m <= kMxMaxM; m++) {
    const int W = 2 * m + 2;
    for (int n0 = 2 * m + 3; n0 < 80; n0++)
      for (int ra = 0; ra < n0; ra++)
        for (int p = ra; p <= ra + mx_ring(W); p++) {
          const int c = mx_plane(p, m, n0);
          if (c < 0 || c >= n0 || (c + m - p) % n0) {
            if (bad++ < 4) std::printf("m=%d n0=%d cell %d plane %d: %d\n", m, n0, ra, p, c);
          }
        }
  }
  for (int n = 5; n < 300; n++)
    for (int nb = 1; nb <= n; nb++)
      for (int c = 0; c < n; c++) {
        const int b = mx_bin(c, n, nb);
        if (b < 0 || b >= nb || c < mx_lo(b, n, nb) || c >= mx_lo(b + 1, n, nb)) bad++;
      }
  return bad != 0;
}
"""


def test_planes_stay_in_the_grid(tmp_path):
    src = tmp_path / "planes.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "planes"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "nfft_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
