// The LDS planes of the standard scheme's marches (kernels_std.hip): the tiles'
// sizes and where a level's rows and columns lie.  Plain C++, so that the
// kernels' reads and writes can be held against the planes on the host.
#pragma once

namespace icaradv {

constexpr int NWAVE = 8;  // waves of a block

// The planes of a field: NR levels of ROWS rows from row -RB on, columns -W..
// 63 + E of the tile, QC words per row
template <int W_, int E_, int RB_, int ROWS_, int NR_>
struct Plane {
    static constexpr int W = W_, E = E_, RB = RB_, ROWS = ROWS_, NR = NR_;
    static constexpr int QC = 64 + W + E, SIZE = ROWS * QC, WORDS = NR * SIZE;
    static constexpr int XH = W + E;  // columns beside a row's 64 lanes
    static constexpr int at(int r, int c) { return (r + RB) * QC + c + W; }
    // plane of level k (k >= -NR)
    static constexpr int level(int k) { return (k + NR) % NR * SIZE; }
};

// k_std_stage: TJ rows of a tile, wave w the RW rows from RW w on; the planes
// hold the stencils' halo rows -HH .. TJ+HH-1
template <int H, int V, int RW>
struct StagePlanes {
    static constexpr int HH = (H + 1) / 2, LA = (V + 1) / 2, TJ = NWAVE * RW;
    using P = Plane<HH, HH - 1, HH, TJ + 2 * HH, V == 1 ? 2 : V>;
};

// k_std_limit: wave w the RW rows from RW w - 1 on.  P, the stage state: rows
// -HH-1 .. TJ-3+HH.  B, the base state and dumb_q: rows -2 .. TJ-1, of which
// the last is never written: the last wave reads its last row's north
// neighbour like every other, into a bound that no wind selects.
template <int H, int V, int RW>
struct LimitPlanes {
    static constexpr int HH = (H + 1) / 2, LA = (V + 1) / 2, TJ = NWAVE * RW;
    static constexpr int LROWS = TJ - 3;  // rows written
    using P = Plane<HH, HH - 1, HH + 1, TJ + 2 * HH - 1, V == 1 ? 2 : V>;
    using B = Plane<1, 0, 2, TJ + 2, 2>;
};

}  // namespace icaradv
