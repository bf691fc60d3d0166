// Rules of the feature pass that a host compiler can check (plain C++; constexpr functions serve device
// code too).
#pragma once

namespace nsc {

// The 2 x 2 cells that the feature pass walks for a box of bw x bh pixels: cw a row, ch rows.  A box
// without pixels (a label that the image does not hold: maxx < minx or maxy < miny) has none: its labels
// would be read from addresses clamped into an empty range.
struct CellWalk {
    int cw, ch;
};
constexpr CellWalk cell_walk(int bw, int bh) { return bw > 0 && bh > 0 ? CellWalk{bw + 1, bh + 1} : CellWalk{1, 0}; }

}  // namespace nsc
