"""The tiles of the marching kernels (csrc/march_tiles.hpp), compiled for the
host: every cell belongs to one at least."""
import subprocess

import pytest

from conftest import REPO

CHECK = r"""
#include <cstdio>
#include <initializer_list>
#include "march_tiles.hpp"

// Tiles of every width up to `most`: from column 0 on, none further from the
// next than it is wide, the last one at (spread: exactly at) the row's end.
int main() {
  int bad = 0;
  for (int v : {2, 4, 8})
    for (int rim : {1, 2, 3, 4}) {
      for (int n0 = 16; n0 <= 40000; n0 += n0 < 20000 ? 1 : 7) {
        const int w = sth::kYmOut * v, tiles = (n0 + w - 1) / w;
        const sth::YmTiles t = sth::ymarch_tiles(n0, tiles, v, rim);
        bool ok = t.first(0, v) == 0;
        for (int b = 1; b < tiles; ++b) {
          const int d = t.first(b, v) - t.first(b - 1, v);
          ok = ok && d > 0 && d <= w && (!t.spread || d >= rim * v);
        }
        const int end = t.first(tiles - 1, v) + w;
        ok = ok && (t.spread ? end == n0 : end >= n0);
        if (!ok && ++bad <= 5) std::printf("v %d rim %d n0 %d\n", v, rim, n0);
      }
    }
  std::printf("%d bad\n", bad);
  return bad != 0;
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiles")

    def go(code):
        (d / "check.cpp").write_text(code)
        subprocess.run(["g++", "-std=c++17", "-O1", f"-I{REPO / 'stencils.jl_amd' / 'csrc'}", str(d / "check.cpp"),
                        "-o", str(d / "check")], check=True)
        return subprocess.run([str(d / "check")], capture_output=True, text=True)

    return go


def test_column_tiles_cover_the_row(run):
    r = run(CHECK)
    assert r.returncode == 0, r.stdout
