// cells.h -- the cell grid of a neighbour-list build (nlist.hip).
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>

struct CellGrid {
  int n[3];                      // cells in each reciprocal direction
  int reach[3];                  // partners lie within +-reach cells
  int total() const { return n[0] * n[1] * n[2]; }
};

// Most cells of a grid: 256 an atom up to 2^24, four an atom beyond, and 16,384 for
// the fewest.  A build clears and scans its cells and holds 8 bytes for each:
// nothing at 16,384, some 60 us and 128 MB at 2^24; 108 atoms in 1000 A at a reach
// of 9 A made 3.7e7 and builds of 48 ms (60 us with the limit), and from 430 reaches
// a side on their number no longer fits an int.  Coarser cells would cost more where
// atoms sit close in a wide box, candidates by the cube of their width (a droplet of
// 4,000 atoms builds in 82 us in a box of 100 reaches, 75 in one of 20).
inline double cell_limit(int natm) {
  const double n = natm;
  return std::max({16384.0, 4.0 * n, std::min(256.0 * n, 16777216.0)});
}

// Cells for partners within rmax between planes W[d] apart: of a third of rmax
// where at least 7 of them fit (partners within +-3 cells), else of a half (5,
// +-2), else of rmax (+-1); 1e-9 margin against rounding of the wrapped
// coordinates.  Coarser where that is more than cell_limit: cells of a half, of
// rmax, then wider by the same factor in every direction.
inline CellGrid choose_cells(const double W[3], double rmax, int natm) {
  const double limit = cell_limit(natm);
  CellGrid g{};
  double k[3];
  auto product = [&] { return k[0] * k[1] * k[2]; };
  for (int most = 3; most >= 1; --most) {
    for (int d = 0; d < 3; ++d) {
      for (g.reach[d] = most; g.reach[d] > 1; --g.reach[d])
        if (std::floor(W[d] * g.reach[d] / (rmax * (1.0 + 1e-9))) >= 2 * g.reach[d] + 1) break;
      k[d] = std::max(1.0, std::floor(W[d] * g.reach[d] / (rmax * (1.0 + 1e-9))));
    }
    if (product() <= limit) break;
  }
  // (a direction that is down to one cell leaves the rest to the others)
  while (product() > limit) {
    const double f = std::min(0.999, std::cbrt(limit / product()));
    for (double& x : k) x = std::max(1.0, std::floor(x * f));
  }
  for (int d = 0; d < 3; ++d) g.n[d] = (int)k[d];
  return g;
}
