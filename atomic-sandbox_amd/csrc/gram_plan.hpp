// How the Gram S^T U splits an m x q product over tiles and chunks of points, and the partial sums that this takes. Host
// code without HIP, so that it can be checked without a GPU.
#pragma once
#include <algorithm>
#include <cstddef>

#include "lira.h"

namespace lira {

// A tile is RB x CB blocks of 16 x 16 outputs. SHARE: it is the whole product and U begins with S, so the blocks that are
// both operands are loaded once and those below S^T S's diagonal are not computed.
constexpr int gram_loaded(int RB, int CB, bool SHARE) { return SHARE ? CB : RB + CB; }
constexpr int gram_computed(int RB, int CB, bool SHARE) { return RB * CB - (SHARE ? RB * (RB - 1) / 2 : 0); }
// waves of a workgroup
constexpr int gram_waves(int RB, int CB, bool SHARE) { return !SHARE ? 4 : RB * CB <= 6 && CB <= 3 ? 16 : 8; }
// whether the accumulators and `each` registers a loaded block fit what the waves leave a lane, 128 or 256
constexpr bool gram_fits(int RB, int CB, bool SHARE, int each) {
    return 8 * gram_computed(RB, CB, SHARE) + each * gram_loaded(RB, CB, SHARE) <=
           (gram_waves(RB, CB, SHARE) == 16 ? 124 : 240);
}
// How a lane loads a 16-column block (GramLoad in kernels_grid.hip). QUAD: four consecutive points of one column. PAIR: 16
// bytes of each of two columns, so that a load instruction takes 128 bytes of a column instead of 64; it needs two column
// pointers a lane, 28 registers a block with both units in flight. PAIR2: two of those a unit, 44 registers.
enum GramLoads { GRAM_QUAD, GRAM_PAIR, GRAM_PAIR2 };
constexpr bool gram_has(int RB, int CB, bool SHARE, int esize, int loads) {
    if (loads == GRAM_PAIR) return gram_fits(RB, CB, SHARE, 28);
    if (loads == GRAM_PAIR2) return esize == 8 && SHARE && gram_waves(RB, CB, SHARE) == 8 && gram_fits(RB, CB, SHARE, 44);
    return true;
}
// loads of a column in a unit, and the unit's points
constexpr int gram_depth(int RB, int CB, int esize, int loads) {
    return loads == GRAM_PAIR2 || (loads == GRAM_QUAD && esize == 4 && RB + CB <= 5) ? 2 : 1;
}
constexpr int gram_unit(int depth, int esize, int loads) { return depth * (loads == GRAM_QUAD ? 16 : 128 / esize); }

// The tiling of an m x q product: nr x nc tiles of RB x CB 16 x 16 blocks (the blocks split evenly, at most 3 x 6 in f32
// or where the one tile shares its operands, else 3 x 4: the accumulators and two units of operands fill 256 registers. In
// f32 without sharing 3 x 6 spills 69 more, and reads each column fewer times: 138 x 276 on 160^3 5.70 ms, 6.32 with 3 x 4;
// 96 x 192 on 95^3 533 us and 509) and the chunks of points. A product of one shared tile takes one workgroup per CU, 16
// waves (4 per SIMD, up to 128 registers) or 8; several tiles take two 4-wave workgroups per CU, so that the tiles that
// S^T S's symmetry empties or thins leave room for others. The partials of one product stay within GRAM_PARTIALS doubles (lira_gram_noalloc's fixed
// array) whenever one chunk's do.
struct GramPlan {
    int RB, CB, nr, nc, chunks, loads;
    bool share;
    long chunk;
};
constexpr long GRAM_PARTIALS = (long)(LIRA_NOALLOC_SCRATCH_BYTES / sizeof(double));
// sym: U's first m columns are S's
inline GramPlan gram_plan(int m, int q, long N, int esize, bool sym) {
    GramPlan g;
    const int R = (m + 15) / 16, C = (q + 15) / 16;
    g.nr = (R + 2) / 3;
    g.RB = (R + g.nr - 1) / g.nr;
    g.nr = (R + g.RB - 1) / g.RB;
    g.share = sym && g.nr == 1 && C <= 6;  // R <= C, for q >= m
    const int most = esize == 4 || g.share ? 6 : 4;
    g.nc = (C + most - 1) / most;
    g.CB = (C + g.nc - 1) / g.nc;
    g.nc = (C + g.CB - 1) / g.CB;
    // PAIR, where it fits, in f64 for more columns than the 256 MiB cache holds (24 x 48 on 95^3 86 -> 75 us; 16 x 32 on
    // 64^3 20 -> 22), in f32 for more than 32 columns a multiple of 8 MiB apart; one block of columns (f64) or two (f32)
    // gained nothing. PAIR2 in f64 from 185^3 on. GramLoad has both sides.
    g.loads = GRAM_QUAD;
    if (gram_has(g.RB, g.CB, g.share, esize, GRAM_PAIR) &&
        (esize == 8 ? g.CB > 1 && q * N * 8 >= 256L << 20 : g.CB > 2 && N * 4 % (8L << 20) == 0))
        g.loads = gram_has(g.RB, g.CB, g.share, esize, GRAM_PAIR2) && N >= 6L << 20 ? GRAM_PAIR2 : GRAM_PAIR;
    long want = std::max(1L, (g.share ? 256L : 512L) / (g.nr * g.nc));
    want = std::max(1L, std::min(want, GRAM_PARTIALS / ((long)m * q)));
    const long unit = gram_unit(gram_depth(g.RB, g.CB, esize, g.loads), esize, g.loads);
    g.chunk = ((N + want - 1) / want + unit - 1) / unit * unit;
    // on small grids, 64 points and a unit for a quarter of the waves: fewer partials to allocate, write and add up
    g.chunk = std::max({g.chunk, 64L, gram_waves(g.RB, g.CB, g.share) / 4 * unit});
    g.chunks = (int)((N + g.chunk - 1) / g.chunk);
    return g;
}

// the partials of one product
inline size_t gram_partials(int m, int q, long N, int esize, bool sym) {
    return (size_t)gram_plan(m, q, N, esize, sym).chunks * m * q;
}

// The partials that suffice for every product of at most m x q columns. A smaller product can need more of them than a
// larger one (f32, U beginning with S: 81 x 162 takes 128 chunks, 243 x 486 takes 14, and 128 * 81 * 162 > 14 * 243 *
// 486), so a buffer that serves several shapes is sized by this: a plan has at most 512 chunks of at least 16 points,
// and more than one only while they stay within GRAM_PARTIALS.
inline size_t gram_partials_bound(int m, int q, long N) {
    const long mq = (long)m * q, chunks = std::min(512L, (N + 15) / 16);
    return (size_t)std::max(mq, std::min(GRAM_PARTIALS, chunks * mq));
}

}  // namespace lira
