// The strip kernel's blocks and which of them a grid takes (host code, no HIP:
// the choice is tested on the CPU).
#pragma once

#include <algorithm>
#include <cstdint>

namespace lmh {

// Grid-stencil geometry of H for the strip kernel (strip.hip): site
// i = x * ly + y on an lx x ly grid, every stored entry of a row being the
// diagonal or one of the four grid neighbours (y +- 1, x +- 1; across the
// edges when px / py).  A strip is s consecutive sites of one x column
// (y0 .. y0 + s - 1), a thread owns the strips of bx neighbouring x columns
// (the last strip or block overlaps its neighbour when s does not divide ly,
// or bx lx), a workgroup `cols` columns of P.
struct StripGeom {
    int lx = 0, ly = 0;
    int lyp = 0;                // LDS length of bx x columns (bx * ly rounded up to odd)
    int px = 0, py = 0;         // periodic along x / y
    int s = 0;                  // sites per strip (0: H is not a grid stencil)
    int bx = 0;                 // x columns per thread
    int q = 0;                  // strips per x column
    int nt = 0;                 // strips of a column of P = lx * q (strip k of x column x: k * lx + x)
    int nthr = 0;               // threads per column of P
    int threads = 0;            // workgroup size
    int cols = 0;               // columns of P per workgroup
    int region = 0;             // LDS entries per column (the last holds 0)
};

constexpr int kStripThreads = 512;      // 8 waves of 256 VGPRs per CU: one workgroup of 512, ..., eight of 64
constexpr int kStripLdsBytes = 163840;
// blocks of x columns by sites: B(bx, s)
#define LMH_STRIP_SHAPES(B) B(1, 20) B(2, 10) B(2, 8) B(2, 6) B(2, 5) B(2, 4) B(4, 4)
struct StripShape {
    int bx, s;
};
constexpr StripShape kStripShapes[] = {
#define LMH_STRIP_SHAPE(BX, S) {BX, S},
    LMH_STRIP_SHAPES(LMH_STRIP_SHAPE)
#undef LMH_STRIP_SHAPE
};
// a block with inner sites does not publish them: its neighbours must not
// read them, so blocks may not overlap nor end early
constexpr bool strip_whole(int bx, int s) { return bx > 2 && s > 2; }

// a grid in blocks of one shape, without the workgroup
inline bool strip_blocks(int64_t lx, int64_t ly, const StripShape &sh, StripGeom *g) {
    if (sh.bx > lx || sh.s > ly) return false;
    if (strip_whole(sh.bx, sh.s) && (lx % sh.bx || ly % sh.s)) return false;
    const int64_t nbx = (lx + sh.bx - 1) / sh.bx, q = (ly + sh.s - 1) / sh.s;
    if (nbx * q > kStripThreads) return false;
    g->lx = (int)lx;
    g->ly = (int)ly;
    g->lyp = (int)((sh.bx * ly) | 1);
    g->bx = sh.bx;
    g->s = sh.s;
    g->q = (int)q;
    g->nt = (int)(lx * q);
    g->nthr = (int)(nbx * q);
    g->region = (int)(nbx * g->lyp + 1);
    return 16 * (int64_t)g->region <= kStripLdsBytes;
}

// How often the LDS serves 16 lanes in turn that read a site each (mean over
// the first wavefront's): lanes whose places agree mod 16 sites meet in the
// same banks.  Blocks side by side are a run of odd pitch apart; a lattice of
// few x columns has them above each other, S sites apart.
inline double strip_conflict(const StripGeom &g) {
    const int nbx = (g.lx + g.bx - 1) / g.bx;
    int turns = 0, groups = 0;
    for (int w = 0; w < std::min(g.nthr, 64); w += 16, ++groups) {
        int slots[16], places[16], count[16] = {};
        const int lanes = std::min(16, g.nthr - w);
        for (int l = 0; l < lanes; ++l) {
            const int k = (w + l) / nbx, b = (w + l) - k * nbx;
            const int x0 = std::min(b * g.bx, g.lx - g.bx), r = x0 / g.bx;
            places[l] = r * g.lyp + (x0 - r * g.bx) * g.ly + std::min(k * g.s, g.ly - g.s);
            slots[l] = places[l] % 16;
            bool again = false;                          // (the same place is one read)
            for (int m = 0; m < l; ++m) again = again || places[m] == places[l];
            if (!again) ++count[slots[l]];
        }
        turns += *std::max_element(count, count + 16);
    }
    return (double)turns / groups;
}

// The cost of a shape: the rounds of workgroups a CU takes (256 CUs of 8 waves),
// each a constant (barriers, latencies, launch), the sites it moves and its
// waves' sites per thread (a wave takes its SIMD's time whether or not the
// others have one), these dearer for large blocks (their diagonal is streamed),
// where S does not divide ly (a term in one phase), for strips of one column
// (42 LDS reads per 20 sites instead of 24) and by the bank conflicts, most
// for blocks 8 sites apart.  Fitted to a step's launches (K = 7 or 8 twice) of
// seven shapes on 247 grids between 2 x 64 and 1000 x 4: the shape it takes is
// 1.7 % behind the best one in the mean, against 7.9 % for a cost without the
// moved sites, the one-phase terms and the conflicts (a step 5 % faster in the
// mean, ladders of 2 x 1000 .. 2 x 4000 1.7 to 2 times).  us per step: 37 x 23
// 2 x 4 33.6, 2 x 8 40.4; 61 x 42 2 x 6 186, 2 x 10 268; 100 x 100 2 x 10 2365,
// 1 x 20 2672; 2 x 2000 2 x 5 407, 1 x 20 414, 2 x 8 776; 5 x 1000 1 x 20 658,
// 2 x 6 730; 340 x 5 2 x 5 158, 2 x 4 218 (their rows shared by two blocks).
// Sets the workgroup size and its columns of P.
inline double strip_cost(StripGeom *g) {
    const int64_t n = (int64_t)g->lx * g->ly;
    const int sites = g->bx * g->s;
    const double f = (sites > 12 ? 1.18 : 1.0) * (g->ly % g->s && g->bx < 4 ? 1.21 : 1.0) * (g->bx == 1 ? 1.28 : 1.0) *
                     (1.0 + std::max(0.0, strip_conflict(*g) - 2.0) * (g->s == 8 ? 0.43 : 0.14));
    double best = 1e300;
    for (int threads = (g->nthr + 63) / 64 * 64; threads <= kStripThreads; threads += 64) {
        const int64_t cols = std::min<int64_t>(threads / g->nthr, kStripLdsBytes / (16 * (int64_t)g->region));
        if (cols < 1) continue;
        const int64_t groups = (n + cols - 1) / cols;
        const int64_t fit = std::min<int64_t>(kStripThreads / threads, kStripLdsBytes / (16 * g->region * cols));
        const int64_t per_cu = std::min<int64_t>(fit, (groups + 255) / 256);
        const int64_t rounds = (groups + 256 * per_cu - 1) / (256 * per_cu);
        const int64_t waves = (per_cu * (threads / 64) + 3) / 4 * 4;
        const double cost = (double)rounds * (53.0 + 0.0135 * (double)(n * cols * per_cu) + (double)(waves * sites) * f);
        if (cost >= best) continue;
        best = cost;
        g->threads = threads;
        g->cols = (int)cols;
    }
    return best;
}

// 2 x 5 is for what two workgroups a CU hold (600 x 5: 485 us, the general
// kernel 345)
inline bool strip_shape_fits(const StripGeom &g) { return g.s != 5 || g.nthr <= kStripThreads / 2; }

// the block shape, workgroup size and columns per workgroup of an lx x ly grid
inline bool strip_shape(int64_t lx, int64_t ly, StripGeom *g) {
    double best = 1e300;
    StripGeom t = *g;
    for (const StripShape &sh : kStripShapes) {
        if (!strip_blocks(lx, ly, sh, &t) || !strip_shape_fits(t)) continue;
        const double cost = strip_cost(&t);
        if (cost >= best) continue;
        best = cost;
        *g = t;
    }
    return best < 1e300;
}

// columns of P in a batch's workgroup of 512 threads
inline int strip_batch_cols(const StripGeom &g) {
    return std::min(kStripThreads / g.nthr, (int)(kStripLdsBytes / (16 * (int64_t)g.region)));
}

// The block shape of a grid's members in a batch, where every workgroup has 512
// threads and every term runs in one phase: the least cost per column of P of
// an otherwise idle CU, fitted to uniform batches of seven shapes on 72 grids
// (0.5 % behind the best in the mean).  The solo shape was up to twice as slow
// there (us per step, N x members ~ 30000: 35 x 35 2 x 5 979, 2 x 8 1145;
// 25 x 100 1 x 20 1920, 2 x 6 2095; 2 x 300 2 x 6 468, 2 x 4 634; 2 x 1000
// 2 x 10 1395, 2 x 8 2756; 64 x 40 4 x 4 1777, 2 x 10 2144).
inline bool strip_batch_shape(int64_t lx, int64_t ly, StripGeom *g) {
    const int64_t n = lx * ly;
    double best = 1e300;
    StripGeom t = *g;
    for (const StripShape &sh : kStripShapes) {
        if (!strip_blocks(lx, ly, sh, &t) || !strip_shape_fits(t)) continue;
        const int64_t cols = strip_batch_cols(t);
        if (cols < 1) continue;
        const int sites = t.bx * t.s;
        const int64_t waves = ((t.nthr * cols + 63) / 64 + 3) / 4 * 4;
        const double f = (t.bx == 4 ? 1.13 : sites == 16 ? 1.30 : sites == 20 ? 1.33 : 1.0) * (t.bx == 1 ? 1.11 : 1.0) *
                         (1.0 + std::max(0.0, strip_conflict(t) - 2.0) * (t.s == 8 ? 0.39 : 0.23));
        const double cost = (64.0 + 0.028 * (double)(n * cols) + (double)(waves * sites) * f) * (double)((n + cols - 1) / cols);
        if (cost >= best) continue;
        best = cost;
        *g = t;
    }
    if (best < 1e300) strip_cost(g);        // (the workgroups of its launches outside the batch)
    return best < 1e300;
}

}  // namespace lmh
