"""Addresses of the band DFT along an axis, walked on the host: the header that the kernel takes
them from is compiled with the host compiler, and every load that any lane of any tile makes stays
inside the tensor, wide loads at aligned addresses, for column counts that do and do not fill the
last tile of 64; lanes of existing columns load their own."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "holoflow_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "axis_columns.hh"

template <int ESZ, bool VEC> void walk(long long outer, int n, long long inner) {
  const long long cols = outer * inner, bytes = outer * n * inner * ESZ;
  const long long width = VEC ? 4 * ESZ : ESZ;  // bytes of one access
  for (long long tile = 0; tile < (cols + 63) / 64; ++tile)
    for (int lane = 0; lane < 16; ++lane) {
      hfx::AxisColumns<ESZ, VEC> a;
      a.init(tile, lane, cols, n, inner);
      for (int t = 0; t < a.N; ++t)
        for (int j = 0; j < n; ++j) {
          const long long at = a.off[t] + j * a.step;
          const long long c = a.column(tile, lane, t), own = ((c / inner * n + j) * inner + c % inner) * ESZ;
          const bool bad = at < 0 || at + width > bytes || (VEC && at % (width < 16 ? width : 16) != 0) ||
                           (c < cols && at != own);
          if (bad) {
            std::printf("esz %d vec %d outer %lld n %d inner %lld: column %lld sample %d reads [%lld, %lld) of %lld bytes\n",
                        ESZ, VEC, outer, n, inner, c, j, at, at + width, bytes);
            std::exit(1);
          }
        }
    }
}

template <int ESZ> void sizes(long long outer, int n, long long inner) {
  walk<ESZ, false>(outer, n, inner);
  if (inner % 4 == 0) walk<ESZ, true>(outer, n, inner);
}

int main() {
  const int ns[] = {1, 2, 3, 9};
  for (long long outer = 1; outer <= 3; ++outer)
    for (int n : ns)
      for (long long inner = 1; inner <= 200; ++inner) {
        sizes<2>(outer, n, inner);
        sizes<4>(outer, n, inner);
        sizes<8>(outer, n, inner);
      }
  sizes<4>(1, 64, 300 * 764);
  return 0;
}
"""


def test_every_load_of_the_axis_dft_stays_inside_the_tensor(tmp_path):
    src = tmp_path / "walk.cpp"
    src.write_text(MAIN)
    exe = tmp_path / "walk"
    subprocess.run(["g++", "-std=c++20", "-O1", "-w", "-D__host__=", "-D__device__=", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
