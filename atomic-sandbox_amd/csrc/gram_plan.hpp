// How the Gram S^T U splits an m x q product over tiles and chunks of points, and the partial sums that this takes. Host
// code without HIP, so that it can be checked without a GPU.
#pragma once
#include <algorithm>
#include <cstddef>

#include "lira.h"

namespace lira {

// The tiling of an m x q product: nr x nc tiles of RB x CB 16 x 16 blocks (the blocks split evenly, at most 3 x 6 in f32
// or where the one tile shares its operands, else 3 x 4: the accumulators and two units of operands fill 256 registers)
// and the chunks of points. A product of one shared tile takes one workgroup per CU, 16 waves (4 per SIMD, up to 128
// registers) or 8; several tiles take two 4-wave workgroups per CU, so that the tiles that S^T S's symmetry empties or
// thins leave room for others. The partials of one product stay within GRAM_PARTIALS doubles (lira_gram_noalloc's fixed
// array) whenever one chunk's do.
struct GramPlan {
    int RB, CB, nr, nc, H, chunks;
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
    g.H = esize == 4 && g.RB + g.CB <= 5 ? 2 : 1;
    long want = std::max(1L, (g.share ? 256L : 512L) / (g.nr * g.nc));
    want = std::max(1L, std::min(want, GRAM_PARTIALS / ((long)m * q)));
    const long unit = 16 * g.H;
    g.chunk = ((N + want - 1) / want + unit - 1) / unit * unit;
    g.chunks = (int)((N + g.chunk - 1) / g.chunk);
    return g;
}

// the partials of one product of m x q columns
inline size_t gram_partials_needed(int m, int q, long N) {
    // the precisions, and U beginning with S or not, may split a product differently
    int chunks = 0;
    for (int esize : {4, 8})
        for (bool sym : {false, true}) chunks = std::max(chunks, gram_plan(m, q, N, esize, sym).chunks);
    return (size_t)chunks * m * q;
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
