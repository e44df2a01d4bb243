// Which kernel advances an iteration of N steps, and in which launches: by
// estimates of what each way takes, in microseconds of an MI355X.  Plain C++,
// with no HIP in it.
//
// An iteration ends with single steps (one launch per step) and may run the
// steps before them in launches of up to G steps each, as many launches as
// leave the buffers alternating as step by step (their number has the parity
// of their steps).  A launch of fewer steps than G still marches through all
// G stages.  So few steps, or arrays of few rows or columns, whose rims are
// most of what a launch computes, may be better off with shorter launches or
// with single steps alone.
//
// The estimates follow what was measured on 14 shapes from 64^2 to 8000 x
// 6000 (rows of 16 to 2^20 cells), four element types, three folds and three
// boundaries, each within about a quarter: 4096^2 f32 Laplacian, Wrap: a
// single step 21 us (estimate 25), a launch of two steps 31 (33), of eight
// 46 (48); 131072 x 16: 5.8 (6.9), 6.6 (7.1) and 27 (32).
#pragma once

#include "march_tiles.hpp"
#include "stencils_hip.h"

namespace sth {

// A kernel of several steps per launch: its most steps, the time of a launch
// of so many, and the share of it that a launch of (almost) none takes.
struct StepKernel {
  int64_t gens;
  double full, idle;
  constexpr double launch(int64_t g) const {
    return g == gens ? full : full * (idle + (1.0 - idle) * static_cast<double>(g) / static_cast<double>(gens));
  }
};

// The launches of an iteration: `multi` launches of at most G steps, then
// `singles` single steps.
struct StepLaunches {
  int64_t multi, singles;
  double time;
};

// Launches of at most G steps for `gens` steps: the fewest of their parity.
constexpr int64_t march_launches(int64_t gens, int64_t G) {
  const int64_t f = (gens + G - 1) / G;
  return f + ((f ^ gens) & 1);
}

// All launches take G steps but the last four, which share the rest: steps of
// launch i of f, with `left` steps to go from it on.
constexpr int64_t march_share(int64_t i, int64_t f, int64_t left, int64_t G) {
  return i + 4 < f ? G : (left + (f - i) - 1) / (f - i);
}

constexpr StepLaunches march_split(int64_t steps, int64_t singles, double single, const StepKernel& k) {
  const int64_t gens = steps - singles, f = march_launches(gens, k.gens), full = f > 4 ? f - 4 : 0;
  double t = static_cast<double>(singles) * single + static_cast<double>(full) * k.full;
  int64_t left = gens - full * k.gens;
  for (int64_t i = full; i < f; ++i) {
    const int64_t g = march_share(i, f, left, k.gens);
    t += k.launch(g);
    left -= g;
  }
  return StepLaunches{f, singles, t};
}

// The cheapest launches of `steps` steps with `k`, of `least` single steps or
// up to three more.
constexpr StepLaunches march_cheapest(int64_t steps, int64_t least, double single, const StepKernel& k) {
  StepLaunches best{0, steps, static_cast<double>(steps) * single};
  for (int64_t s = least; s < least + 4 && s < steps; ++s) {
    const StepLaunches l = march_split(steps, s, single, k);
    if (best.multi == 0 || l.time < best.time) best = l;
  }
  return best;
}

// The launch that refreshes the halo of `rows` rows: cells at the rows' ends
// are a line of memory each (262144 rows: 14 us).
constexpr double march_halo(int64_t rows, double launch) { return launch + 4e-5 * static_cast<double>(rows); }

// ------------------------------------------------------- 2-D iterations

// What the estimates need of a 2-D call.
struct MarchCall {
  int64_t n0, n1;
  int dtype, op, L, bc;
  bool rows16;     // rows start on 16-byte boundaries
  bool catalogue;  // the single step is a build-time kernel
  bool halo;       // each single step refreshes a halo first
  int cell() const {
    return dtype == STH_BF16 || dtype == STH_F16 || dtype == STH_I16 || dtype == STH_U16 ? 2
           : dtype == STH_F64 || dtype == STH_I64 || dtype == STH_U64                    ? 8
                                                                                         : 4;
  }
  bool is_float() const { return dtype == STH_F32 || dtype == STH_F64 || dtype == STH_BF16 || dtype == STH_F16; }
  double megabytes() const { return 2e-6 * static_cast<double>(n0 * n1 * cell()); }  // read and written by a step

  // Vector operations per cell and step, in issue slots of a 4-byte one.
  double ops() const {
    const bool extreme = op == STH_OP_MAX || op == STH_OP_MIN, wide = cell() == 8;
    double c = op == STH_OP_LAPLACIAN ? L + 2.4 : op == STH_OP_MEAN ? L + 10.0 : extreme ? (is_float() ? 4.0 : 0.75) * L
               : op == STH_OP_KERNELPRODUCT ? 2.0 * L : L + 0.5;
    if (wide && !extreme) c *= 1.5;
    if (cell() == 2) c += 3.0;
    if (bc == STH_REFLECT) c += wide ? 6.0 : 3.0;  // the fix-ups of the rims
    if (bc == STH_REMOVE) c += wide ? 2.0 : 1.0;
    return c;
  }

  // One step in a launch of its own: 3.5 to 5 us of launch, then memory (6.5
  // TB/s from the Infinity Cache, 5.2 past it), of which rows that leave lanes
  // idle or start on any byte reach less.
  double single() const {
    const int v = 16 / cell();
    const int64_t lanes = (n0 + v - 1) / v;
    int64_t row = 8;
    while (row < 64 && row < lanes) row *= 2;
    const double mb = megabytes(), full = lanes < row ? static_cast<double>(row) / static_cast<double>(lanes) : 1.0;
    double t = mb < 256.0 ? 4.3 + mb / 6.5 * full * (rows16 ? 1.0 : 1.5) : mb / 5.2;
    if (cell() == 2) {
      const double u = mb < 256.0 ? 8.0 + mb / 4.2 * full * (rows16 ? 1.0 : 1.4) : mb / 3.6;
      if (u > t) t = u;
    }
    return (catalogue ? t : 1.25 * t) + (halo ? march_halo(n1, 5.0) : 0.0);
  }

  // ymarch_kernel built for G steps per launch.  A row step of a wave issues
  // G V ops() operations, 4 cycles each at 2.4 GHz.
  StepKernel march(int gens, int64_t cus) const {
    const int v = 16 / cell();
    const YmGrid g = ymarch_grid(n0, n1, v, gens, cus);
    const double c = ops(), step = gens * v * c / 600.0, traffic = megabytes() / 4.6;
    double t = 0;
    if (gens == kYmShortGens) {
      const int64_t own = g.rows < n1 ? g.rows : n1, steps = (own + 2 * gens + kYmAhead - 1) / kYmAhead * kYmAhead;
      const double waves = static_cast<double>(g.tx * ((n1 + g.rows - 1) / g.rows)) / static_cast<double>(4 * cus) + 0.4;
      const double issue = (waves > 1.0 ? waves : 1.0) * static_cast<double>(steps) * step * 1.15;
      t = 3.5 + (issue > traffic ? issue : traffic);
    } else {
      const double units = ym_units(g, gens, cus);
      t = 1.5 + (units * step > traffic ? units * step : traffic);
    }
    // rows of part vectors that are not spread load and store cell by cell,
    // which a short launch cannot hide
    if (n0 % v != 0 && !ymarch_tiles(static_cast<int>(n0), static_cast<int>(g.tx), v, (gens + v - 1) / v).spread)
      t *= gens == kYmShortGens ? 1.7 : 1.2;
    // an idle stage moves its rows on: few operations a cell, but in 16-bit
    // types registers spill then
    double idle = cell() == 2 || gens == kYmShortGens ? 1.0 : (cell() == 8 ? 7.0 : 4.5) / c + (bc == STH_REMOVE ? 0.3 : 0.0);
    return StepKernel{gens, t, idle < 1.0 ? idle : 1.0};
  }

  // Row steps of a launch in units of a wave's issue time (as ymarch_grid
  // weighs them, but with part rounds).
  static double ym_units(const YmGrid& g, int gens, int64_t cus) {
    const double steps = static_cast<double>(g.rows + 2 * gens), total = static_cast<double>(g.tx * g.ty);
    const double rounds = 0.2 + total / static_cast<double>(2 * cus);
    return steps * (total <= static_cast<double>(cus) ? 1.6 : 2.25 * (rounds > 1.0 ? rounds : 1.0));
  }
};

// How a 2-D iteration of `steps` steps runs: steps per launch of the kernel
// (0: none) and the single steps at its end, `least` at least.
struct MarchChoice {
  int gens;
  int64_t singles;
};

// The long launches are the rule.  Where the estimates say so clearly, short
// launches or single steps replace them: by a tenth for a few steps, a quarter
// for more; at once for large arrays of few rows, where the rims are most of a
// long launch (262144 x 16 f64 mean, Reflect, 33 steps: 688 us with six steps
// per launch, 357 with two).  Arrays of fewer than kYmMinCells rows have the
// short ones only.
inline MarchChoice march_choose(const MarchCall& c, int long_gens, int64_t steps, int64_t least, int64_t cus) {
  const double single = c.single();
  const StepLaunches s = march_cheapest(steps, least, single, c.march(kYmShortGens, cus));
  MarchChoice alt = s.time < static_cast<double>(steps) * single ? MarchChoice{kYmShortGens, s.singles} : MarchChoice{0, steps};
  double alt_time = s.time < static_cast<double>(steps) * single ? s.time : static_cast<double>(steps) * single;
  if (c.n1 < kYmMinCells) return alt;
  const StepKernel k = c.march(long_gens, cus);
  const StepLaunches l = march_cheapest(steps, least, single, k);
  const double margin = c.n1 < 64 && c.n0 * c.n1 >= (int64_t(1) << 20) ? 1.0 : steps <= 8 ? 1.1 : 1.25;
  return alt_time * margin < l.time ? alt : MarchChoice{long_gens, l.singles};
}

// ------------------------------------------------------- 3-D iterations

// How a 3-D star iteration of f32 (or 2-byte, `es`) cells runs: on
// zmarch_kernel with the single steps at its end, or (singles = steps) as it
// would otherwise: in pairs of steps on zmarch2_kernel where the array is
// large enough for it (`pairs`), else in single steps.
//
// A launch of four steps of zmarch_kernel takes its rounds of workgroups times
// their plane steps, 0.35 us each and step (Wrap: 200^3 8.5, 256^3 11.8, 384^3
// 30, 512^3 73.5 us a step; the edge cells of Remove and Reflect make it 0.47
// and 0.5, 2-byte storage 15% more), one of three steps 0.85 of it.
// zmarch2_kernel takes 1.06 us per 10^6 cells and step, 6 at least (f32 Wrap:
// 128^3 6.1, 200^3 10.0, 256^3 17.5, 384^3 66, 512^3 162 us; 2-byte cells move
// half the bytes and keep it), a single step 5 + 2 per 10^6 cells (32^3 4.8,
// 100^3 7.5, 256^3 32; in launches of four 3.9, 4.5 and 11.8), with a halo the
// launch that refreshes it more, which a `graph` hides for the most part (32^3,
// Reflect: 12 us a step launch by launch, 6 in a graph).
inline int64_t zmarch_singles(int64_t n0, int64_t n1, int64_t n2, int bc, int es, const ZmGrid& grid, bool pairs,
                              bool halo, bool graph, int64_t steps, int64_t least) {
  if (pairs && es != 4) return steps;
  const double mcells = 1e-6 * static_cast<double>(n0) * static_cast<double>(n1) * static_cast<double>(n2);
  const double single = 5.0 + 2.0 * mcells + (es == 4 ? 0.0 : 1.0) + (halo ? march_halo(n1 * n2, graph ? 1.0 : 5.0) : 0.0);
  const double unit = (bc == STH_WRAP ? 0.35 : (bc == STH_REMOVE ? 0.47 : 0.5)) * (es == 4 ? 1.0 : 1.15);
  const StepLaunches star =
      march_cheapest(steps, least, single, StepKernel{kZmGens, kZmGens * unit * static_cast<double>(grid.time), 0.4});
  double other = static_cast<double>(steps) * single;
  if (pairs && steps >= 7) {
    const int64_t units = (steps - 3) / 4;  // pairs of launches
    other = static_cast<double>(steps - 4 * units) * single +
            static_cast<double>(4 * units) * (1.06 * mcells > 6.0 ? 1.06 * mcells : 6.0);
  }
  return star.time < other ? star.singles : steps;
}

}  // namespace sth
