// trsv_tile.hpp -- several Jacobi sweeps per launch on boxes of a grid.
#pragma once

#include "parilu.hpp"

namespace lace {

// Most coupled sweeps of one launch: the halo grows with them on every side
// the factor reads from.
constexpr int kTileC = 4;

// One launch's boxes (sides and halos in rows).
struct TileShape {
  int n, nx, ny, nz;  // the grid
  int bx, by, bz;     // box
  int hx, hy, hz;     // halo on the side the factor reads from (hx a multiple of a unit)
  int ex, ey, ez;     // widened box
  int tx, ty, tz;     // boxes along each axis
  int c;              // coupled sweeps
  int nux;            // units along a line of the widened box
  unsigned mx, my;    // 2^20 / nux and 2^20 / ey, rounded up
};

// Whether `sweeps` Jacobi sweeps of P run on boxes that read the 16-bit
// diagonal form (and no FP32 copy of it).
bool jacobi_tile16(const TriPlan& P, int sweeps);

// Whether `sweeps` Jacobi sweeps of P with the value array val run on boxes:
// a grid with every neighbour present (TriPlan::grid), its diagonal form
// current, byte offsets of a vector within 31 bits, and ahead of one-sweep
// launches there.
template <typename T>
bool jacobi_tile_ready(const TriPlan& P, const T* val, int sweeps);

// c (1..kTileC) coupled sweeps in one launch from yin, or from the first
// sweep's r / diag where yin is null; yout must be neither r nor yin.
template <typename T>
int jacobi_tile(const TriPlan& P, const T* r, const T* yin, T* yout, int c);

}  // namespace lace
