// The integer arithmetic of the matrix products (gemm.hip): which tile a unit is, which part of an
// operand it reads and how many bytes of memory its loads may touch. Nothing here needs a device, so
// that a host program can walk every unit of a product and check each range against its operand
// (tests/gemm_ranges.cpp).
#pragma once

#include <cstdint>

namespace mykfa {

constexpr int kGemmBK = 64;  // K columns per stage
constexpr int kGemmCUs = 256;

constexpr int gemm_min(int a, int b) { return a < b ? a : b; }
constexpr int gemm_max(int a, int b) { return a > b ? a : b; }
constexpr int gemm_round8(int x) { return (x + 7) & ~7; }
constexpr int gemm_stages(int k) { return k > 0 ? (k + kGemmBK - 1) / kGemmBK : 1; }

// One launch's share of a product: tm x tn tiles per batch and split of K, of `side` x `side` launch
// tiles each (2 where a launch takes the last units of a larger tile's list as quarters).
struct GemmGrid {
    int tm, tn, splits, stages;  // K stages per split
    int first_unit;
    bool quarters;
};

struct GemmTile {
    int outer, bidx, m0, n0, kt0, nk;  // outer = batch * splits + split; K stages [kt0, kt0 + nk)
};

// Groups of up to 8 row tiles run down the columns, so the tiles resident on an XCD share its L2's
// panels. bm x bn: the launch's tile.
constexpr GemmTile gemm_tile(const GemmGrid& g, int k, int unit, int bm, int bn) {
    const int quad = g.quarters ? unit & 3 : 0, side = g.quarters ? 2 : 1;
    unit = g.first_unit + (g.quarters ? unit >> 2 : unit);
    const int tiles = g.tm * g.tn, x = unit % tiles;
    const int gsz = 8 * g.tn, grp = x / gsz, in = x % gsz, gm = gemm_min(8, g.tm - grp * 8);
    GemmTile t{};
    t.outer = unit / tiles;
    t.bidx = t.outer / g.splits;
    t.kt0 = t.outer % g.splits * g.stages;
    t.nk = gemm_min(g.stages, gemm_stages(k) - t.kt0);
    t.m0 = ((grp * 8 + in % gm) * side + (quad & 1)) * bm;
    t.n0 = (in / gm * side + (quad >> 1)) * bn;
    return t;
}

// What a tile reads of one operand: `rows` stored rows and `cols` stored columns from the element
// at row `row0`, column `col0`. Its rows or columns of M / N (mn of them in all) begin at r0. A quarter
// can begin past them: it has no rows and reads nothing.
struct GemmPart {
    int row0, col0, rows, cols;
};
template <bool TR>
constexpr GemmPart gemm_part(int mn, int k, int r0, int tile) {
    if (TR) {  // rows of K, columns of M / N
        const int cols = gemm_max(gemm_round8(mn) - r0, 0);
        return GemmPart{0, r0, cols > 0 ? k : 0, cols};
    }
    return GemmPart{r0, 0, gemm_max(gemm_min(mn - r0, tile), 0), gemm_round8(k)};
}
// The same for K stage kt of it: first row and column from the part's, and the bytes from there on that a
// load may touch (a load past them reads zeros).
struct GemmSpan {
    int row, col, bytes;
};
template <bool TR>
constexpr GemmSpan gemm_span(const GemmPart& p, int rs, int kt) {
    const int k0 = kt * kGemmBK;
    if (TR) {
        const int r = gemm_min(p.rows - k0, kGemmBK);
        return GemmSpan{k0, 0, r > 0 ? ((r - 1) * rs + p.cols) * 2 : 0};
    }
    const int left = p.cols - k0;
    return GemmSpan{0, k0, left > 0 && p.rows > 0 ? ((p.rows - 1) * rs + left) * 2 : 0};
}

}  // namespace mykfa
