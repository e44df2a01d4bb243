"""The host side of the multi-step kernels, compiled for the CPU: the tiles of
the marching kernels (csrc/march_tiles.hpp: every cell belongs to one at least),
the launches of an iteration and their choice (csrc/march_cost.hpp), and the
tile shapes of the packed Life kernel (csrc/lifep_shape.hpp)."""
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
        subprocess.run(["g++", "-std=c++17", "-O1", f"-I{REPO / 'stencils.jl_amd' / 'csrc'}",
                        f"-I{REPO / 'include'}", str(d / "check.cpp"),
                        "-o", str(d / "check")], check=True)
        return subprocess.run([str(d / "check")], capture_output=True, text=True)

    return go


def test_column_tiles_cover_the_row(run):
    r = run(CHECK)
    assert r.returncode == 0, r.stdout


ZGRID = r"""
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include "march_tiles.hpp"

using sth::ZmGrid;

// every chunk count that some chunk length gives, the first of the shortest
static ZmGrid walk(int64_t n0, int64_t n1, int64_t n2, int64_t cus) {
  const int64_t gx = (n0 + 55) / 56, gy = (n1 + 55) / 56;
  ZmGrid best{gx, gy, 0, 0};
  for (int64_t c = 1; c <= n2; ++c) {
    const int64_t zc = (n2 + c - 1) / c;
    if ((n2 + zc - 1) / zc != c) continue;
    const int64_t t = (gx * gy * c + cus - 1) / cus * ((zc + 8 + 5) / 6 * 6);
    if (best.tz == 0 || t < best.time) best = ZmGrid{gx, gy, c, t};
  }
  return best;
}

int main() {
  int bad = 0;
  auto one = [&](int64_t n0, int64_t n1, int64_t n2, int64_t cus) {
    const ZmGrid a = sth::zmarch_grid(n0, n1, n2, cus), b = walk(n0, n1, n2, cus);
    if ((a.tx != b.tx || a.ty != b.ty || a.tz != b.tz || a.time != b.time) && ++bad <= 5)
      std::printf("%ld x %ld x %ld on %ld: %ld chunks, %ld, not %ld, %ld\n", long(n0), long(n1), long(n2), long(cus),
                  long(a.tz), long(a.time), long(b.tz), long(b.time));
  };
  for (int64_t n2 = 16; n2 <= 1200; ++n2)
    for (int64_t g = 1; g <= 40; ++g) one(g * 56 - 3, 50, n2, 256);
  std::srand(1);
  for (int i = 0; i < 20000; ++i)
    one(16 + std::rand() % 2000, 16 + std::rand() % 2000, 16 + std::rand() % 3000, i % 3 ? 256 : 32 + std::rand() % 300);
  one(16, 16, 1000000, 256);
  one(3000, 300, 100000, 256);
  long steps = 0;
  const auto t0 = std::chrono::steady_clock::now();
  for (int64_t k = 0; k < 10; ++k) steps += sth::zmarch_grid(16, 16 + k, 1000000 + k, 256).tz;
  const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 10;
  std::printf("%d bad, %ld, %.2f us a search\n", bad, steps, us);
  // (one search over 10^6 chunk counts takes milliseconds)
  return bad != 0 || us > 200.0;
}
"""


def test_plane_chunks_are_the_shortest(run):
    r = run(ZGRID)
    print(r.stdout)
    assert r.returncode == 0, r.stdout


COST = r"""
#include <cstdio>
#include <initializer_list>
#include "march_cost.hpp"

using namespace sth;
static int bad = 0;
static void expect(bool ok, const char* what, long a = 0, long b = 0) {
  if (!ok && ++bad <= 10) std::printf("%s (%ld, %ld)\n", what, a, b);
}
static MarchCall call(int64_t n0, int64_t n1, int dtype, int op, int L, int bc) {
  return MarchCall{n0, n1, dtype, op, L, bc, true, true, false};
}

int main() {
  // the launches of an iteration: all its steps, none longer than G, their number of the parity of their steps
  for (int64_t G : {2, 4, 6, 8})
    for (int64_t least : {1, 2})
      for (int64_t n = 4; n <= 300; ++n) {
        const StepLaunches l = march_cheapest(n, least, 5.0, StepKernel{G, 9.0, 0.5});
        expect(l.singles >= least && l.singles < n, "single steps", G, n);
        const int64_t gens = n - l.singles, f = march_launches(gens, G);
        expect(f == l.multi && (f - gens) % 2 == 0, "launches", G, n);
        int64_t left = gens;
        for (int64_t i = 0; i < f; ++i) {
          const int64_t g = march_share(i, f, left, G);
          expect(g >= 1 && g <= G, "steps of a launch", G, n);
          left -= g;
        }
        expect(left == 0, "steps left", G, n);
      }
  // as measured (us): see march_choose
  expect(march_choose(call(262144, 16, STH_F64, STH_OP_MEAN, 9, STH_REFLECT), 6, 33, 1, 256).gens == 2, "few rows");
  expect(march_choose(call(262144, 16, STH_F32, STH_OP_LAPLACIAN, 4, STH_REMOVE), 8, 7, 1, 256).gens != 8, "few rows, few steps");
  expect(march_choose(call(1 << 21, 8, STH_F32, STH_OP_LAPLACIAN, 4, STH_WRAP), 8, 33, 1, 256).gens == 2, "8 rows");
  expect(march_choose(call(16, 262144, STH_F32, STH_OP_MEAN, 9, STH_WRAP), 6, 33, 1, 256).gens == 0, "few columns");
  const MarchChoice five = march_choose(call(300, 200, STH_F32, STH_OP_MEAN, 9, STH_WRAP), 6, 5, 1, 256);
  expect(five.gens != 6 || five.singles == 2, "five steps: not in two long launches and a single step");
  for (int64_t n : {512, 1024, 2048, 4096, 8192}) {
    expect(march_choose(call(n, n, STH_F32, STH_OP_LAPLACIAN, 4, STH_WRAP), 8, 100, 1, 256).gens == 8, "f32 heat", n);
    expect(march_choose(call(n, n, STH_F64, STH_OP_LAPLACIAN, 4, STH_WRAP), 8, 100, 1, 256).gens == 8, "f64 heat", n);
    expect(march_choose(call(n, n, STH_F32, STH_OP_MEAN, 9, STH_REMOVE), 6, 100, 1, 256).gens == 6, "f32 mean", n);
  }
  // 3-D: three steps in one launch and three single ones, not three launches (64^3 f32, 6 steps: 60 us, 46 before)
  for (int64_t n : {32, 64, 100})
    expect(zmarch_singles(n, n, n, STH_WRAP, 4, zmarch_grid(n, n, n, 256), false, false, false, 6, 1) >= 3, "3-D, six steps", n);
  for (int64_t n : {64, 100, 200, 256, 384})
    expect(zmarch_singles(n, n, n, STH_WRAP, 4, zmarch_grid(n, n, n, 256), n >= 128, false, true, 100, 1) < 8, "3-D, 100 steps", n);
  std::printf("%d bad\n", bad);
  return bad != 0;
}
"""


def test_launches_and_choices(run):
    r = run(COST)
    assert r.returncode == 0, r.stdout


LIFE = r"""
#include <chrono>
#include <cstdio>
#include "lifep_shape.hpp"

using namespace sth;

int main() {
  int bad = 0;
  // more sizes than are remembered, each twice
  for (int64_t i = 0; i < 3000; ++i) {
    const int64_t n0 = 64 + 7 * i, n1 = 3 + (i * i) % 9000;
    const LifepShape a = lifep_shape(n0, n1, i % 2 != 0, 256), b = lifep_shape(n0, n1, i % 2 != 0, 256),
                     c = lifep_search(n0, n1, i % 2 != 0, 256);
    const bool same = a.k == b.k && a.gens == b.gens && a.lpr_shift == b.lpr_shift && a.k == c.k && a.gens == c.gens &&
                      a.lpr_shift == c.lpr_shift;
    // a tile keeps at least one row, a rim word at least the bits it loses
    if (!same || a.gens > kLifepMaxGens || (kLifepWaves << (6 - a.lpr_shift)) * a.k - 2 * a.gens < 1) ++bad;
  }
  const auto t0 = std::chrono::steady_clock::now();
  for (int i = 0; i < 1000; ++i) bad += lifep_shape(1501, 1333, true, 256).k < 1;
  const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 1000;
  std::printf("%d bad, %.2f us a call\n", bad, us);
  return bad != 0 || us > 3.0;  // the search itself takes four times that
}
"""


def test_life_shapes_are_remembered(run):
    r = run(LIFE)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
