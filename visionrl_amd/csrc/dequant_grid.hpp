// How the dequant launch cuts a weight into tiles.  Plain C++: the arithmetic is tested on the host.
#pragma once

namespace {

constexpr int DEQUANT_THREADS = 256;
constexpr int DEQUANT_TILES = 65535;   // row tiles of one launch: what gridDim.y takes; beyond it a call is several

// A row of kwords packed words is cut into `segments` of 1 << tshift words (the power of two that covers it, 256 at
// most); a tile is one segment of `span` rows, `rows` of them per thread.
struct DequantGrid {
    int tshift, segments, rows, span;
    int tiles;   // row tiles
};

inline DequantGrid dequant_grid(int N, int K) {
    DequantGrid g{0, 0, 0, 0, 0};
    const int kwords = K >> 3;
    while (g.tshift < 8 && (1 << g.tshift) < kwords) ++g.tshift;
    g.segments = (int)(((long)kwords + (1 << g.tshift) - 1) >> g.tshift);
    // Four independent rows per thread keep enough loads in flight once the chip is full; below that more, shorter
    // threads are done sooner (512 x 2048: 2.4 us, against 3.2 with four rows and a division for the segment).
    g.rows = (long)N * kwords <= (1L << 18) ? 1 : 4;
    g.span = g.rows * (DEQUANT_THREADS >> g.tshift);
    g.tiles = (int)(((long)N + g.span - 1) / g.span);
    return g;
}

}  // namespace
