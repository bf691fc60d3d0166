// Rules of the watershed's passes that a host compiler can check (plain C++; constexpr functions serve
// device code too).
#pragma once

namespace nsc {

// k_classify's wide path for the four pixels i0 .. i0 + 3 of a plane of N = W * H pixels: it reads the
// markers i0 - 1 .. i0 + 4 and four of the rows above and below, and of the colours (3 bytes a pixel) the
// bytes 3 i0 - 4 .. 3 i0 + 15 and twelve of the rows above and below.  The rows ask for i0 >= W and
// i0 + 3 + W < N, the four bytes that hold the next pixel's colour for i0 + 6 <= N (which a plane of
// width 1 does not get from the rows).
constexpr bool classify_wide(int i0, int W, int N) { return i0 >= W && i0 + 3 + W < N && i0 + 6 <= N; }

}  // namespace nsc
