// Walks the tiles of a matrix product as the GPU does and checks every stage's memory range against the
// operand it reads. Lines of stdin: transposed (0 / 1) mn other k row_stride; the operand is (mn, k)
// rows, or (k, mn) with transposed, and `other` is the product's other dimension. Each is walked as the
// row operand and as the column operand, in tiles of 256, 128 and 64 and in quarters of the 256s, in one
// and in three parts of K. Prints the ranges that leave their operand; exits with 1 if there is one.
#include <cstdio>

#include "../myk_llm_amd/csrc/gemm_tiles.h"

using namespace mykfa;

static long long bad = 0, walked = 0;

template <bool TR>
static void stage(int mn, int k, int rs, int r0, int tile, int kt) {
    const GemmPart p = gemm_part<TR>(mn, k, r0, tile);
    const GemmSpan s = gemm_span<TR>(p, rs, kt);
    const int rows = TR ? k : mn, cols = TR ? mn : k;
    const long long from = ((long long)(p.row0 + s.row) * rs + p.col0 + s.col) * 2;
    const long long end = ((long long)(rows - 1) * rs + gemm_round8(cols)) * 2;
    ++walked;
    if (s.bytes < 0 || (s.bytes > 0 && from + s.bytes > end)) {
        if (++bad <= 20)
            std::printf("%s mn %d k %d row stride %d: tile at %d, stage %d: %d bytes from %lld of %lld\n", TR ? "TR" : "rows", mn,
                        k, rs, r0, kt, s.bytes, from, end);
    }
}

template <bool TR>
static void walk(int mn, int other, int k, int rs) {
    for (int as_row = 0; as_row < 2; ++as_row)
        for (int size = 256; size >= 64; size /= 2)
            for (int quarters = 0; quarters < (size == 256 ? 2 : 1); ++quarters)
                for (int parts = 1; parts <= 3; parts += 2) {
                    const int m = as_row ? mn : other, n = as_row ? other : mn;
                    GemmGrid g{(m + size - 1) / size, (n + size - 1) / size, 1, 0, 0, quarters != 0};
                    g.stages = (gemm_stages(k) + parts - 1) / parts;
                    g.splits = (gemm_stages(k) + g.stages - 1) / g.stages;
                    const int tile = quarters ? size / 2 : size;
                    const int units = g.tm * g.tn * g.splits * (quarters ? 4 : 1);
                    int last = -1;
                    for (int u = 0; u < units; ++u) {
                        const GemmTile t = gemm_tile(g, k, u, tile, tile);
                        const int r0 = as_row ? t.m0 : t.n0;
                        if (t.nk < 1 || t.bidx != 0) {
                            ++bad;
                            std::printf("unit %d of %d: batch %d, %d stages\n", u, units, t.bidx, t.nk);
                        }
                        if (r0 == last) continue;
                        last = r0;
                        for (int kt = t.kt0; kt < t.kt0 + t.nk; ++kt) stage<TR>(mn, k, rs, r0, tile, kt);
                    }
                }
}

int main() {
    int tr, mn, other, k, rs;
    while (std::scanf("%d %d %d %d %d", &tr, &mn, &other, &k, &rs) == 5) {
        if (tr) walk<true>(mn, other, k, rs);
        else walk<false>(mn, other, k, rs);
    }
    std::printf("%lld ranges, %lld outside\n", walked, bad);
    return bad != 0;
}
