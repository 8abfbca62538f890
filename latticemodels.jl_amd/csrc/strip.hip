// Fused Taylor pass for grid-stencil Hamiltonians: the "strip" kernel.
//
// The square lattices of LatticeModels.jl (SquareLattice, site i = x Ly + y,
// src/lattices/bravais/lattice.jl:101-111) give an H whose row i holds the
// diagonal and the four grid neighbours i +- 1 (y +- 1) and i +- Ly (x +- 1),
// across the edges for periodic boundaries.  Under a Landau gauge
// (src/zoo/magneticfields.jl:11-15) a y bond's phase depends on x only and an
// x bond carries none, so along a run of consecutive sites of one x column
// every bond of one direction has the same value.  This kernel uses both
// facts:
//
//   * a thread owns a block of BX x columns by S sites of a column of P and
//     keeps y and x of the Horner recursion in registers; neighbours inside
//     the block are its own registers, so per term only the sites around the
//     block come from LDS, plus one write of each site on its edge;
//   * the block's bond values are registers, read once per launch; so is the
//     diagonal (on-site disorder) of a small block, a large one streams it
//     from L2 a row ahead.
//
// Per Horner term  y <- x + (-i dt / (s k)) H y  the new values of a block's
// edge are published to the column's LDS copy.  Where S divides ly a term
// runs in two phases of rows, each phase's values being published while the
// other computes (a write costs the LDS as much as three reads: published on
// their own before the term, they took a third of it); else the values are
// published, then a term runs (rows that two blocks share would belong to
// different phases).  The column is loaded with gfx950 direct-to-LDS loads
// (global_load_lds 16 B per lane).  A workgroup has as few wavefronts as a
// column needs: 8 wavefronts a CU, in one workgroup at N = 10^4, whose loads
// and stores then only overlap with other CUs' sums, in several at smaller N.
// A step's launch (both sides, K = 8), strips of one column by 12 .. 20 sites
// in workgroups of 512 before, blocks now: N = 100 48 -> 21 us, 851 47 -> 30,
// 1681 144 -> 89, 2304 165 -> 143, 4096 518 -> 491, 6400 1374 -> 1182, 10^4
// 2866 -> 2252.  At N = 10^4 a term takes 4400 cycles per CU (7200 before), of
// which FP64 issue 3020 and LDS 3090; loads and stores take 1.0 ms of the
// launch, 0.68 at the copy rate.
// The workgroup is persistent over its share of the columns.
//
// Whether H qualifies is decided twice: the pattern on the host when the
// geometry is set (strip_detect, which also picks the block shape:
// strip_shape.h), and the values after every H build on the device
// (h_check_kernel: every used bond of a strip's direction equal to the strip's
// value, and that the conjugate of its partner's, bit for bit).  When either
// fails, the fused passes run the kernels of column.hip or fused.hip, so this
// kernel changes speed, never results.  Reference step: src/evolution.jl:73-78 (U P U' with U from
// myexp!, :93-128); the polynomial is the reference's order-K Taylor
// polynomial evaluated in Horner form.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <set>
#include <type_traits>
#include <vector>

#include "lmhip_internal.h"

namespace lmh {

namespace {

constexpr int kStripMaxN = 10240;
constexpr int strip_shape_id(int bx, int s) { return bx * 32 + s; }
// (kStripMaxK: Horner coefficients passed with the launch or read from a
// TaylorOut, lmhip_internal.h)

// one Taylor polynomial p(-i dts H)^reps of a pass
struct StripPoly {
    const double2 *stval;   // [4][nt] bond value per direction: y+, y-, x+, x-
    const double *sdiag;    // [s][nt] diagonal per strip position
    int K;
    int reps;
    double dts;             // dt / s
    double ck[kStripMaxK + 1];  // ck[k] = dts / k for k <= min(K, kStripMaxK)
    const TaylorOut *coef;  // when set: K, reps and ck read from here instead
};

// a device TaylorOut read through the constant address space: wave-uniform
// scalar loads (nothing writes it while a strip launch runs)
typedef __attribute__((address_space(4))) const TaylorOut ConstTaylorOut;

// global memory by pointers read from memory (a batch member's): told apart
// from LDS, whose counter their loads and stores would otherwise hold up
typedef double vec2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) vec2 GlobalVec2;
typedef __attribute__((address_space(1))) const vec2 ConstGlobalVec2;
typedef __attribute__((address_space(1))) const double ConstGlobalDouble;

struct StripArgs {
    StripGeom g;
    StripPoly poly[2];      // applied to each column in this order
    int npoly;              // 1, or 2: the second step's first side fused onto the first's second
    const double2 *X;
    double2 *Y;
    int64_t ld;
    int64_t ncols;
    int n;
    int64_t nprog;          // workgroups (a multiple of 8)
    int64_t stagger;        // start delay (shader cycles) of every other group of 8 workgroups
    int xreal;              // batched kernel: the member's x bonds are real
    const TaylorOut *guard; // when set: the launch runs only if strip_coef_ok(*guard, guard_xreal)
    int guard_xreal;
};

__device__ __forceinline__ void cmac(double2 &acc, double2 h, double2 v) {
    acc.x = fma(h.x, v.x, acc.x);
    acc.x = fma(-h.y, v.y, acc.x);
    acc.y = fma(h.x, v.y, acc.y);
    acc.y = fma(h.y, v.x, acc.y);
}

// MI355X deals workgroups round-robin to its 8 XCDs: logical workgroup
// numbers run consecutively on one XCD, so the conjugate-transposed stores of
// neighbouring columns (one 128-byte line holds 8 of them) meet in one L2.
__device__ __forceinline__ int64_t strip_xcd_order(int64_t b, int64_t nprog) {
    const int64_t per = nprog / kNumXCD;
    return (b % kNumXCD) * per + b / kNumXCD;
}

// LDS place of x column x of a column of P: bx x columns to a run of pitch
// lyp (odd, so that the lanes of a wave, whose blocks sit a run apart, read
// from distinct banks)
__device__ __forceinline__ int strip_run(const StripGeom &g, int x) {
    const int r = x / g.bx;
    return r * g.lyp + (x - r * g.bx) * g.ly;
}

// direct-to-LDS loads of the column group starting at jb: one wave
// instruction per 64 sites of a run
__device__ __forceinline__ void strip_dma(const StripArgs &a, double2 *lds, int64_t jb, int wave, int lane) {
    const StripGeom &g = a.g;
    int64_t ldg = a.ld;
    asm volatile("" : "+s"(ldg));
    const int len = g.bx * g.ly;
    const int nch = (len + 63) >> 6, nrun = (g.lx + g.bx - 1) / g.bx;
    const int per_col = nrun * nch;
    const int npair = g.cols * per_col;
    const int waves = (int)blockDim.x >> 6;
    for (int p = wave; p < npair; p += waves) {
        const int gg = p / per_col;
        const int rem = p - gg * per_col;
        const int r = rem / nch, ch = rem - r * nch;
        const int64_t jj = jb + gg;
        const int e = ch * 64 + lane;
        const int i = r * len + e;
        if (jj < a.ncols && e < len && i < a.n) {
            const double2 *src = a.X + jj * ldg + i;
            __builtin_amdgcn_global_load_lds(
                (const void *)src,
                (__attribute__((address_space(3))) void *)(lds + gg * g.region + r * g.lyp + ch * 64), 16, 0, 0);
        }
    }
}

// plain result of the column group starting at jb from its LDS copy: the
// inverse of strip_dma, one 1 KB contiguous store per wave instruction
__device__ __forceinline__ void strip_store(const StripArgs &a, const double2 *lds, int64_t jb, int wave, int lane) {
    const StripGeom &g = a.g;
    int64_t ldg = a.ld;
    asm volatile("" : "+s"(ldg));
    const int len = g.bx * g.ly;
    const int nch = (len + 63) >> 6, nrun = (g.lx + g.bx - 1) / g.bx;
    const int per_col = nrun * nch;
    const int npair = g.cols * per_col;
    const int waves = (int)blockDim.x >> 6;
    for (int p = wave; p < npair; p += waves) {
        const int gg = p / per_col;
        const int rem = p - gg * per_col;
        const int r = rem / nch, ch = rem - r * nch;
        const int64_t jj = jb + gg;
        const int e = ch * 64 + lane;
        const int i = r * len + e;
        if (jj < a.ncols && e < len && i < a.n) {
            const double2 v = lds[gg * g.region + r * g.lyp + e];
            ((GlobalVec2 *)a.Y)[jj * ldg + i] = vec2{v.x, v.y};
        }
    }
}

// acc += h v for a complex h, or for a real h (XR: h.y == 0, two FMAs)
template <bool XR>
__device__ __forceinline__ void hmac(double2 &acc, double2 h, double2 v) {
    if constexpr (XR) {
        acc.x = fma(h.x, v.x, acc.x);
        acc.y = fma(h.x, v.y, acc.y);
    } else {
        cmac(acc, h, v);
    }
}

constexpr int kNoSite = 1 << 30;

// A thread's place in the column group: its block of BX x columns by S sites
// and the LDS positions of its columns and neighbours.
template <int BX>
struct StripThread {
    int slot, tl, x0, y0, skx, sky;              // skx, sky: columns and rows shared with the block before
    int cb[BX], xl, xr;                          // own columns at y0; the columns left and right of the block
    int lo, hi;                                  // from cb: the sites below and above the block (kNoSite: absent)
    int zero;                                    // an entry that holds 0
    bool act;
};

template <int BX, int S>
__device__ __forceinline__ StripThread<BX> strip_thread(const StripArgs &a) {
    const StripGeom &g = a.g;
    StripThread<BX> p;
    const int t = threadIdx.x;
    p.slot = t / g.nthr;                         // column of the workgroup this thread works on
    p.act = p.slot < g.cols;
    const int th = p.act ? t - p.slot * g.nthr : 0;        // idle threads mirror thread 0 (no writes)
    const int rb = p.act ? p.slot * g.region : 0;
    const int nbx = (g.lx + BX - 1) / BX;
    const int k = th / nbx, bx = th - k * nbx;
    p.x0 = min(bx * BX, g.lx - BX);
    p.skx = bx * BX - p.x0;
    p.y0 = min(k * S, g.ly - S);
    p.sky = k * S - p.y0;
    p.tl = k * g.lx + p.x0;                      // the block's first strip
    p.zero = rb + g.region - 1;
#pragma unroll
    for (int i = 0; i < BX; ++i) p.cb[i] = rb + strip_run(g, p.x0 + i) + p.y0;
    // an absent x neighbour reads the own column (its bond value is 0), an
    // absent y neighbour the zero entry
    const int xr = p.x0 + BX < g.lx ? p.x0 + BX : (g.px ? 0 : g.lx - 1);
    const int xl = p.x0 > 0 ? p.x0 - 1 : (g.px ? g.lx - 1 : 0);
    p.xr = rb + strip_run(g, xr) + p.y0;
    p.xl = rb + strip_run(g, xl) + p.y0;
    p.lo = p.y0 > 0 ? -1 : (g.py ? g.ly - 1 : kNoSite);
    p.hi = p.y0 + S < g.ly ? S : (g.py ? S - g.ly : kNoSite);
    return p;
}

// a block's bond values: y + 1 of each column (y - 1: its conjugate), and the
// x bonds between its columns and to the left and right of it, each as the
// value that multiplies the site to the right of it (for the site to the left:
// its conjugate)
template <int BX>
struct StripBonds {
    double2 hy[BX], hx[BX + 1];
};
template <int BX, bool XR>
__device__ __forceinline__ StripBonds<BX> strip_bonds(const double2 *stval, int nt, int tl) {
    ConstGlobalVec2 *sv = (ConstGlobalVec2 *)stval;
    StripBonds<BX> b;
#pragma unroll
    for (int i = 0; i < BX; ++i) {
        const vec2 u = sv[tl + i], h = sv[2 * nt + tl + i];
        b.hy[i] = make_double2(u.x, u.y);
        b.hx[i + 1] = make_double2(h.x, XR ? 0.0 : h.y);
    }
    const vec2 h = sv[3 * nt + tl];
    b.hx[0] = make_double2(h.x, XR ? 0.0 : -h.y);
    return b;
}

// One column group of a strip pass, its columns already in LDS (with the
// zero slot set).  TOUT: the result is written conjugate-transposed
// (Y[s, j] = conj(y_s)), else plainly; XR: the x bonds are real (Landau
// gauge, no field).  TWO: a.npoly polynomials in turn, each with its bond
// values loaded when it starts (else one, its bond values in p1).  At the end
// the next group (na, njb, when next) is loaded into LDS with its zero slot,
// ready for the next call.
// PHASES: a term in two phases, which needs S to divide ly (rows shared by two
// blocks would belong to different phases); else in one, its input published
// before it.
template <int BX, int S, bool TOUT, bool XR, bool TWO, bool PHASES>
__device__ __forceinline__ void strip_group(const StripArgs &a, const StripThread<BX> &p, const StripBonds<BX> &p1,
                                            double2 *lds, int64_t jb, const StripArgs &na, int64_t njb, bool next) {
    const StripGeom &g = a.g;
    const int t = threadIdx.x;
    const bool act = p.act;
    const int wave = t >> 6, lane = t & 63;
    const int64_t j = jb + p.slot;
    double2 xr[S][BX], yv[S][BX];
#pragma unroll
    for (int m = 0; m < S; ++m)
#pragma unroll
        for (int i = 0; i < BX; ++i) {
            xr[m][i] = lds[p.cb[i] + m];
            yv[m][i] = xr[m][i];
        }
    for (int ph = 0; ph < (TWO ? a.npoly : 1); ++ph) {
    // this polynomial's parameters (selected, not indexed: a dynamic index
    // into the argument block would copy it to scratch memory)
    const double2 *stv = ph ? a.poly[1].stval : a.poly[0].stval;
    const double *sdg = ph ? a.poly[1].sdiag : a.poly[0].sdiag;
    const TaylorOut *pcf = ph ? a.poly[1].coef : a.poly[0].coef;
    ConstTaylorOut *cf = (ConstTaylorOut *)pcf;
    const int PK = pcf ? cf->K : (ph ? a.poly[1].K : a.poly[0].K);
    const int preps = pcf ? cf->reps : (ph ? a.poly[1].reps : a.poly[0].reps);
    const double pdts = ph ? a.poly[1].dts : a.poly[0].dts;
    StripBonds<BX> b = p1;
    if constexpr (TWO) {
        // the opaque copy keeps the addresses from being hoisted out of the
        // loops
        int tq = p.tl;
        asm volatile("" : "+v"(tq));
        b = strip_bonds<BX, XR>(stv, g.nt, tq);
    }
    // a small block keeps its diagonal in registers, a large one streams it
    // from L2 a row ahead
    constexpr bool DREG = BX * S <= 12;
    double dr[DREG ? S : 1][BX];
    if constexpr (DREG) {
#pragma unroll
        for (int m = 0; m < S; ++m)
#pragma unroll
            for (int i = 0; i < BX; ++i) dr[m][i] = ((ConstGlobalDouble *)sdg)[m * g.nt + p.tl + i];
    }
    // One Horner term in two phases of rows: the edge rows (E first and E
    // last ones), then the middle ones.  While a phase computes, the other's
    // rows go to LDS, where a neighbour reads them: the middle rows of the
    // term before during the edge phase, the new edge rows during the middle
    // one.  Every value read in a phase was written a barrier ago and is
    // overwritten a barrier later, so the writes (as dear as three reads)
    // cost no phase of their own, and one LDS copy does.
    // UP: the rows of each segment upwards, else downwards.  A site's new
    // value takes the register its neighbour's old value leaves free, one row
    // over in the sweep's direction; alternating the direction puts the
    // values back in place after two terms instead of moving them all at the
    // loop's end.  Each site's arithmetic is the same either way.
    auto term = [&](int kk, bool publish_first, auto up) {
        constexpr bool UP = decltype(up)::value;
        constexpr int E = S / 4 > 0 ? S / 4 : 1, NE = 2 * E, NM = S - NE, NM_ = NM > 0 ? NM : 1;
        constexpr auto row = [](int r) {
            const int u = !PHASES || r < E ? r : (r < NE ? S - NE + r : r - E);
            return UP ? u : S - 1 - u;
        };
        // (an idle thread holds and writes what thread 0 does)
        auto publish = [&](int m) {
#pragma unroll
            for (int i = 0; i < BX; ++i)
                if (m == 0 || m == S - 1 || i == 0 || i == BX - 1)
                    lds[p.cb[i] + m] = yv[m][i];
        };
        const double c = pcf ? cf->ck[kk]
                             : (kk <= kStripMaxK ? (ph ? a.poly[1].ck[kk] : a.poly[0].ck[kk]) : pdts / (double)kk);
        // opaque copy: keeps the diagonal addresses from being hoisted out of
        // the term loop into registers
        int ntq = g.nt;
        asm volatile("" : "+s"(ntq));
        ConstGlobalDouble *sd = (ConstGlobalDouble *)sdg + p.tl;
        constexpr int kAhead = BX == 1 ? 4 : (BX == 2 && S <= 8 ? 3 : (PHASES ? 1 : 2));
        double dv[S][BX];
#pragma unroll
        for (int r = 0; r < (DREG ? S : kAhead); ++r)
#pragma unroll
            for (int i = 0; i < BX; ++i) dv[row(r)][i] = DREG ? dr[row(r)][i] : sd[row(r) * ntq + i];
        if (!PHASES && publish_first) {
            // the previous term's reads are done; publish this term's input
            __syncthreads();
#pragma unroll
            for (int m = 0; m < S; ++m) publish(m);
            __syncthreads();
        }
        // the sites outside the block, below and above
        auto outside = [&](bool above, int i) {
            const int o = above ? p.hi : p.lo;
            return lds[o == kNoSite ? p.zero : p.cb[i] + o];
        };
        double2 back[BX], keep[2][BX], endv[BX];         // keep: the old edge rows next to the middle ones, by segment
        double2 av[S], bv[S];
#pragma unroll
        for (int i = 0; i < BX; ++i) back[i] = outside(!UP, i);
#pragma unroll
        for (int r = 0; r < S; ++r) {
            const int m = row(r);
            if (r == 0 || (PHASES && r == NE)) {
                av[m] = lds[p.xl + m];
                bv[m] = lds[p.xr + m];
            }
            // a segment's first row: the old row behind it
            if (PHASES && r == E) {
#pragma unroll
                for (int i = 0; i < BX; ++i) {
                    back[i] = NM > 0 ? yv[UP ? S - E - 1 : E][i] : keep[0][i];
                }
            }
            if (r == (PHASES ? (E > 2 ? NE - 2 : NE - 1) : (BX > 1 ? S - 1 : S - 2))) {
#pragma unroll
                for (int i = 0; i < BX; ++i) endv[i] = outside(UP, i);
            }
            if (PHASES && r == NE) {
#pragma unroll
                for (int i = 0; i < BX; ++i) back[i] = keep[0][i];
            }
            if (r + 1 < (PHASES && r < NE ? NE : S)) {
                av[row(r + 1)] = lds[p.xl + row(r + 1)];
                bv[row(r + 1)] = lds[p.xr + row(r + 1)];
            }
            double2 left = av[m];
#pragma unroll
            for (int i = 0; i < BX; ++i) {
                if (!DREG && r + kAhead < S) dv[row(r + kAhead < S ? r + kAhead : r)][i] = sd[row(r + kAhead < S ? r + kAhead : r) * ntq + i];
                const double2 cur = yv[m][i];
                const int mn = UP ? m + 1 : m - 1;           // the row ahead
                const double2 ahead = r == (PHASES ? NE : S) - 1 ? endv[i]
                                      : PHASES && r == S - 1     ? keep[1][i]
                                                                 : yv[mn < 0 ? 0 : (mn < S ? mn : S - 1)][i];
                if (PHASES && r == E - 1) keep[0][i] = cur;
                if (PHASES && r == E) keep[1][i] = cur;
                const double2 nyp = UP ? ahead : back[i];     // site y + 1 (old value)
                const double2 nym = UP ? back[i] : ahead;     // site y - 1 (old value)
                const double2 right = i + 1 < BX ? yv[m][i + 1] : bv[m];
                double2 acc = make_double2(dv[m][i] * cur.x, dv[m][i] * cur.y);
                cmac(acc, b.hy[i], nyp);
                cmac(acc, make_double2(b.hy[i].x, -b.hy[i].y), nym);
                hmac<XR>(acc, b.hx[i + 1], right);
                hmac<XR>(acc, make_double2(b.hx[i].x, -b.hx[i].y), left);
                back[i] = cur;
                left = cur;
                // y_new = x + (-i c) acc
                yv[m][i] = make_double2(fma(c, acc.y, xr[m][i].x), fma(-c, acc.x, xr[m][i].y));
                // (opaque: the sum stays in this phase instead of moving, with
                // its operands, to where the value is next used)
                asm volatile("" : "+v"(yv[m][i].x), "+v"(yv[m][i].y));
                if (PHASES && i == 0) {
                    // the other phase's rows, a row's share at a time
                    if (r < NE) {
#pragma unroll
                        for (int q = r * NM / NE; q < (r + 1) * NM / NE; ++q) publish(E + q);
                    } else {
#pragma unroll
                        for (int q = (r - NE) * NE / NM_; q < (r - NE + 1) * NE / NM_; ++q) publish(row(q));
                    }
                }
                // one site at a time: bounds the live neighbour values
                __builtin_amdgcn_sched_barrier(0);
            }
            if (PHASES && (r == NE - 1 || r == S - 1)) __syncthreads();
        }
        if (PHASES && NM == 0) {
#pragma unroll
            for (int m = 0; m < S; ++m) publish(m);
            __syncthreads();
        }
    };
    for (int rr = 0; rr < preps; ++rr) {
        int kk = PK;
        for (; kk >= 2; kk -= 2) {
            term(kk, ph > 0 || rr > 0 || kk != PK, std::true_type{});
            term(kk - 1, true, std::false_type{});
        }
        // an odd term count ends on a downward sweep (an upward one here
        // needs more registers than the kernel has)
        if (kk == 1) term(1, ph > 0 || rr > 0 || PK != 1, std::false_type{});
        // the next repetition (or polynomial) acts on this one's result
        if (rr + 1 < preps || (TWO && ph + 1 < a.npoly)) {
#pragma unroll
            for (int m = 0; m < S; ++m)
#pragma unroll
                for (int i = 0; i < BX; ++i) xr[m][i] = yv[m][i];
        }
    }
    }
    // the last term's LDS reads are done (or the column's own, when there is
    // no term)
    __syncthreads();
    if constexpr (TOUT) {
        // the next column group loads while this one's results leave from
        // registers: Y[s, j] = conj(y_s), a column of the result is a row of Y
        if (next) strip_dma(na, lds, njb, wave, lane);
        if (act && j < a.ncols) {
            int64_t ldq = a.ld;
            asm volatile("" : "+s"(ldq));
#pragma unroll
            for (int i = 0; i < BX; ++i) {
                GlobalVec2 *yo = (GlobalVec2 *)a.Y + ((int64_t)(p.x0 + i) * g.ly + p.y0) * ldq + j;
#pragma unroll
                for (int m = 0; m < S; ++m) {
                    if (i >= p.skx && m >= p.sky) *yo = vec2{yv[m][i].x, -yv[m][i].y};
                    yo += ldq;
                }
            }
        }
    } else {
        // plain: the results go through the LDS copy so that each wave store
        // covers 64 consecutive sites (a thread's own 16-byte stores would be
        // one request each); then the next group loads
        if (act) {
#pragma unroll
            for (int m = 0; m < S; ++m)
#pragma unroll
                for (int i = 0; i < BX; ++i) lds[p.cb[i] + m] = yv[m][i];
        }
        __syncthreads();
        strip_store(a, lds, jb, wave, lane);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __syncthreads();
        if (next) strip_dma(na, lds, njb, wave, lane);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // the next group's zero slots (past its sites: the loads leave them alone)
    if (next && t < na.g.cols) lds[(t + 1) * na.g.region - 1] = make_double2(0.0, 0.0);
    __syncthreads();
}

template <int BX, int S, bool TOUT, bool XR, bool TWO, bool PHASES>
__global__ void __launch_bounds__(kStripThreads) strip_kernel(StripArgs a) {
    extern __shared__ double2 lds[];
    // a polynomial the host did not see: nothing to do unless it is the one
    // the launch was chosen for (the host tests the same and redoes the step)
    if (a.guard && !strip_coef_ok(*a.guard, a.guard_xreal != 0)) return;
    const StripGeom &g = a.g;
    const int t = threadIdx.x;
    const int wave = t >> 6, lane = t & 63;
    int64_t r = strip_xcd_order(blockIdx.x, a.nprog);
    int64_t jb = r * g.cols;
    // every other group of 8 workgroups (neighbouring columns on one XCD)
    // starts about half a column period later: the workgroups then do not
    // all load and store at the same time nor all compute at the same time
    if (a.stagger > 0 && ((r >> 3) & 1)) {
        const int64_t t0 = (int64_t)clock64();
        while ((int64_t)clock64() - t0 < a.stagger) __builtin_amdgcn_s_sleep(16);
    }
    if (t < g.cols) lds[(t + 1) * g.region - 1] = make_double2(0.0, 0.0);
    if (jb < a.ncols) strip_dma(a, lds, jb, wave, lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const StripThread<BX> p = strip_thread<BX, S>(a);
    StripBonds<BX> b{};
    if constexpr (!TWO) b = strip_bonds<BX, XR>(a.poly[0].stval, g.nt, p.tl);
    while (jb < a.ncols) {
        const int64_t rn = r + a.nprog, jbn = rn * g.cols;
        strip_group<BX, S, TOUT, XR, TWO, PHASES>(a, p, b, lds, jb, a, jbn, jbn < a.ncols);
        r = rn;
        jb = jbn;
    }
}

// the batch member that owns work unit u (ustart: prefix sums of the
// members' column-group counts)
__device__ __forceinline__ int strip_member_of(const int64_t *__restrict__ ustart, int nm, int64_t u) {
    int lo = 0, hi = nm - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (ustart[mid] <= u) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template <bool TOUT, bool XR>
__device__ __forceinline__ void strip_group_s(const StripArgs &a, double2 *lds, int64_t jb, const StripArgs &na,
                                              int64_t njb, bool next) {
    switch (strip_shape_id(a.g.bx, a.g.s)) {
#define LMH_STRIP_GROUP(BX, S)                                                                             \
    case strip_shape_id(BX, S): {                                                                          \
        const StripThread<BX> p = strip_thread<BX, S>(a);                                                  \
        const StripBonds<BX> b = strip_bonds<BX, XR>(a.poly[0].stval, a.g.nt, p.tl);                       \
        strip_group<BX, S, TOUT, XR, false, false>(a, p, b, lds, jb, na, njb, next);                       \
        break;                                                                                             \
    }
        LMH_STRIP_SHAPES(LMH_STRIP_GROUP)
#undef LMH_STRIP_GROUP
        default: break;
    }
}

// Many independent density matrices (batch members of any grid size and
// strip length) in one persistent launch: the work units are the members'
// column groups, concatenated; workgroup r takes units r, r + nprog, ...
// (consecutive units, i.e. neighbouring columns of one member, on one XCD).
template <bool TOUT>
__global__ void __launch_bounds__(kStripThreads) batched_strip_kernel(const StripArgs *__restrict__ members,
                                                                      const int64_t *__restrict__ ustart, int nm,
                                                                      int64_t nunits, int64_t nprog) {
    extern __shared__ double2 lds[];
    const int t = threadIdx.x;
    const int wave = t >> 6, lane = t & 63;
    int64_t u = strip_xcd_order(blockIdx.x, nprog);
    if (u >= nunits) return;
    int m = strip_member_of(ustart, nm, u);
    int64_t jb = (u - ustart[m]) * members[m].g.cols;
    if (t < members[m].g.cols) lds[(t + 1) * members[m].g.region - 1] = make_double2(0.0, 0.0);
    strip_dma(members[m], lds, jb, wave, lane);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    while (u < nunits) {
        const int64_t un = u + nprog;
        const int mn = un < nunits ? strip_member_of(ustart, nm, un) : m;
        const int64_t jbn = un < nunits ? (un - ustart[mn]) * members[mn].g.cols : 0;
        if (members[m].xreal)
            strip_group_s<TOUT, true>(members[m], lds, jb, members[mn], jbn, un < nunits);
        else
            strip_group_s<TOUT, false>(members[m], lds, jb, members[mn], jbn, un < nunits);
        u = un;
        m = mn;
        jb = jbn;
    }
}

// Copies for a deferred pass whose polynomial the host has not seen: the
// strip values and the order record, only when the launch it follows ran
// (the same test as its guard), so that a launch that did nothing leaves the
// earlier pass's copies in place.
__global__ void __launch_bounds__(256) strip_snapshot_kernel(const double2 *__restrict__ sv, const double *__restrict__ sd,
                                                             int64_t nsv, int64_t nsd, const TaylorOut *__restrict__ coef,
                                                             int xreal, double2 *__restrict__ sv_out,
                                                             double *__restrict__ sd_out,
                                                             TaylorOut *__restrict__ coef_out) {
    if (!strip_coef_ok(*coef, xreal != 0)) return;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nsv; e += stride) sv_out[e] = sv[e];
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nsd; e += stride) sd_out[e] = sd[e];
    if (blockIdx.x == 0 && threadIdx.x == 0) *coef_out = *coef;
}

// the dynamic-LDS attribute, once per device and instantiation
template <int BX, int S, bool T, bool XR, bool TWO, bool PHASES>
hipError_t strip_attr() {
    static std::atomic<uint64_t> done{0};
    return once_per_device(done, [] {
        return hipFuncSetAttribute((const void *)strip_kernel<BX, S, T, XR, TWO, PHASES>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kStripLdsBytes);
    });
}

template <int BX, int S, bool T, bool XR, bool TWO, bool PHASES>
hipError_t launch_s(const StripArgs &a, size_t lds, hipStream_t st) {
    hipError_t e = strip_attr<BX, S, T, XR, TWO, PHASES>();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((strip_kernel<BX, S, T, XR, TWO, PHASES>), dim3((unsigned)a.nprog), dim3((unsigned)a.g.threads), lds,
                       st, a);
    return hipGetLastError();
}

// two polynomials in one launch only with conjugate-transposed stores
template <int BX, int S, bool PHASES>
hipError_t launch_sx(bool tout, bool xr, const StripArgs &a, size_t lds, hipStream_t st) {
    if (a.npoly > 1)
        return xr ? launch_s<BX, S, true, true, true, PHASES>(a, lds, st) : launch_s<BX, S, true, false, true, PHASES>(a, lds, st);
    if (tout)
        return xr ? launch_s<BX, S, true, true, false, PHASES>(a, lds, st) : launch_s<BX, S, true, false, false, PHASES>(a, lds, st);
    return xr ? launch_s<BX, S, false, true, false, PHASES>(a, lds, st) : launch_s<BX, S, false, false, false, PHASES>(a, lds, st);
}

template <int BX, int S, bool PHASES>
hipError_t prepare_sx() {
    hipError_t e = strip_attr<BX, S, true, true, false, PHASES>();
    if (e == hipSuccess) e = strip_attr<BX, S, true, false, false, PHASES>();
    if (e == hipSuccess) e = strip_attr<BX, S, false, true, false, PHASES>();
    if (e == hipSuccess) e = strip_attr<BX, S, false, false, false, PHASES>();
    if (e == hipSuccess) e = strip_attr<BX, S, true, true, true, PHASES>();
    if (e == hipSuccess) e = strip_attr<BX, S, true, false, true, PHASES>();
    return e;
}

hipError_t dispatch_s(bool tout, bool xr, const StripArgs &a, size_t lds, hipStream_t st) {
    switch (strip_shape_id(a.g.bx, a.g.s)) {
#define LMH_STRIP_CASE(BX, S) \
    case strip_shape_id(BX, S):                                                                       \
        return a.g.ly % S ? launch_sx<BX, S, strip_whole(BX, S)>(tout, xr, a, lds, st) : launch_sx<BX, S, true>(tout, xr, a, lds, st);
        LMH_STRIP_SHAPES(LMH_STRIP_CASE)
#undef LMH_STRIP_CASE
        default: return hipErrorInvalidValue;
    }
}

// H's row pattern as an lx x ly grid (site i = x ly + y)?  Fills the slot of
// each direction of each site.
bool try_grid(const int32_t *col, int64_t n, int zmax, int64_t lx, int64_t ly, int px, int py, int32_t *sslot) {
    std::fill(sslot, sslot + 4 * n, -1);
    for (int64_t i = 0; i < n; ++i) {
        const int64_t x = i / ly, y = i % ly;
        int64_t nb[4];
        nb[0] = y + 1 < ly ? i + 1 : (py ? i - (ly - 1) : -1);
        nb[1] = y > 0 ? i - 1 : (py ? i + ly - 1 : -1);
        nb[2] = x + 1 < lx ? i + ly : (px ? i - (lx - 1) * ly : -1);
        nb[3] = x > 0 ? i - ly : (px ? i + (lx - 1) * ly : -1);
        for (int u = 0; u < zmax; ++u) {
            const int64_t q = (int64_t)u * n + i;
            const int32_t c = col[q];
            if (c < 0) continue;
            int d = 0;
            while (d < 4 && nb[d] != c) ++d;
            if (d == 4 || sslot[d * n + i] >= 0) return false;
            sslot[d * n + i] = (int32_t)q;
        }
        for (int d = 0; d < 4; ++d)
            if (nb[d] >= 0 && sslot[d * n + i] < 0) return false;
    }
    return true;
}

bool has_entry(const int32_t *col, int64_t n, int zmax, int64_t i, int64_t j) {
    for (int u = 0; u < zmax; ++u)
        if (col[(int64_t)u * n + i] == j) return true;
    return false;
}

}  // namespace

bool strip_detect(const int32_t *col, int64_t n, int zmax, StripGeom *g, int32_t *sslot) {
    *g = StripGeom{};
    if (n < 9 || n > kStripMaxN || zmax < 1 || zmax > 4) return false;
    std::set<int64_t> cands;
    for (int64_t q = 0; q < (int64_t)zmax * n; ++q) {
        if (col[q] < 0) continue;
        const int64_t d = std::llabs((int64_t)col[q] - q % n);
        for (int64_t c : {d, d + 1, n - d})
            if (c >= 3 && c < n && n % c == 0) cands.insert(c);
    }
    for (int64_t ly : cands) {
        const int64_t lx = n / ly;
        if (lx < 2) continue;
        // the edges are periodic when their wrap-around bond is there
        const int py = ly >= 3 && has_entry(col, n, zmax, ly - 1, 0);
        const int px = lx >= 3 && has_entry(col, n, zmax, (lx - 1) * ly, 0);
        if (!try_grid(col, n, zmax, lx, ly, px, py, sslot)) continue;
        if (ly < 4 || !strip_shape(lx, ly, g)) continue;
        g->px = px;
        g->py = py;
        return true;
    }
    std::fill(sslot, sslot + 4 * n, -1);
    return false;
}

namespace {

StripPoly strip_poly(const double2 *stval, const double *sdiag, double dt_over_s, int K, int reps) {
    StripPoly q{};
    q.stval = stval;
    q.sdiag = sdiag;
    q.K = K;
    q.reps = reps;
    q.dts = dt_over_s;
    for (int k = 0; k <= kStripMaxK; ++k) q.ck[k] = k ? dt_over_s / (double)k : 0.0;
    return q;
}

StripArgs strip_args(const DevHam &h, const double2 *X, double2 *Y, int64_t ld, int64_t ncols, double dt_over_s,
                     int K, int reps) {
    StripArgs a{};
    a.g = h.sg;
    a.poly[0] = strip_poly(h.stval, h.sdiag, dt_over_s, K, reps);
    a.npoly = 1;
    a.X = X;
    a.Y = Y;
    a.ld = ld;
    a.ncols = ncols;
    a.n = (int)h.n;
    a.xreal = h.strip_xreal != 0;
    return a;
}

hipError_t device_cus(int *cus) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev);
    return e;
}

}  // namespace

namespace {

// persistent grid, start stagger and LDS size of a strip pass, then the launch
hipError_t launch_args(const DevHam &h, StripArgs &a, int64_t ncols, bool tout, hipStream_t st) {
    const StripGeom &g = h.sg;
    int cus = 0;
    hipError_t e = device_cus(&cus);
    if (e != hipSuccess) return e;
    const int64_t groups = (ncols + g.cols - 1) / g.cols;
    const size_t lds = (size_t)g.cols * g.region * sizeof(double2);
    const int64_t per_cu = std::min<int64_t>(kStripThreads / g.threads, kStripLdsBytes / (int64_t)lds);
    const int64_t np = std::min<int64_t>(groups, per_cu * std::max(cus, 1));
    a.nprog = ((np + kNumXCD - 1) / kNumXCD) * kNumXCD;
    // half a column period in shader cycles (at N = 10^4 in 2 x 10 blocks: 220
    // cycles per site of a block and term, 6 per site of a column for its load
    // and store), when each workgroup has several column groups to do (a step
    // at 100 x 100: 2410 us without, 2370 with it, 2450 with twice as much; at
    // 96 x 96 and below within 1 % of none)
    int64_t terms = 0;
    for (int q = 0; q < a.npoly; ++q) terms += (int64_t)a.poly[q].K * a.poly[q].reps;
    a.stagger = per_cu == 1 && groups >= 4 * a.nprog
                    ? (int64_t)((220.0 * terms * g.bx * g.s + 6.0 * (double)h.n * g.cols) / 2.0)
                    : 0;
    return dispatch_s(tout, a.xreal != 0, a, lds, st);
}

bool strip_shape_ok(const DevHam &h, int64_t ncols, bool tout) {
    const StripGeom &g = h.sg;
    return g.s != 0 && h.n == (int64_t)g.lx * g.ly && (!tout || ncols == h.n);
}

}  // namespace

hipError_t launch_strip(const DevHam &h, const double2 *X, double2 *Y, int64_t ld, int64_t ncols, double dt_over_s,
                        int K, int reps, bool tout, hipStream_t st, const StripPending *second,
                        const TaylorOut *coef) {
    if (!strip_shape_ok(h, ncols, tout) || (second && !tout)) return hipErrorInvalidValue;
    if (ncols == 0) return hipSuccess;
    StripArgs a = strip_args(h, X, Y, ld, ncols, dt_over_s, K, reps);
    a.poly[0].coef = coef;
    a.guard = coef;
    a.guard_xreal = h.strip_xreal != 0;
    if (second) {
        // the previous step's second side first, then this step's first side
        a.poly[1] = a.poly[0];
        a.poly[0] = strip_poly(second->stval, second->sdiag, second->dts, second->K, second->reps);
        a.poly[0].coef = second->coef;
        a.npoly = 2;
        a.xreal = a.xreal && second->xreal;
    }
    return launch_args(h, a, ncols, tout, st);
}

hipError_t launch_strip_pending(const DevHam &h, const StripPending &q, const double2 *X, double2 *Y, int64_t ld,
                                int64_t ncols, bool tout, hipStream_t st) {
    if (!strip_shape_ok(h, ncols, tout)) return hipErrorInvalidValue;
    if (ncols == 0) return hipSuccess;
    StripArgs a = strip_args(h, X, Y, ld, ncols, q.dts, q.K, q.reps);
    a.poly[0].stval = q.stval;
    a.poly[0].sdiag = q.sdiag;
    a.poly[0].coef = q.coef;
    a.xreal = q.xreal;
    return launch_args(h, a, ncols, tout, st);
}

hipError_t launch_strip_snapshot(const DevHam &h, const TaylorOut *coef, bool xreal, double2 *stval, double *sdiag,
                                 TaylorOut *coef_out, hipStream_t st) {
    const int64_t nsv = strip_stval_count(h), nsd = strip_sdiag_count(h);
    const int64_t work = std::max(nsv, nsd);
    const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>((work + 255) / 256, 1024));
    hipLaunchKernelGGL(strip_snapshot_kernel, dim3((unsigned)blocks), dim3(256), 0, st, h.stval, h.sdiag, nsv, nsd,
                       coef, (int)xreal, stval, sdiag, coef_out);
    return hipGetLastError();
}

hipError_t strip_batch_table(const StripMemberDesc *m, int nm, void **d_args, int64_t **d_ustart, int64_t *nunits,
                             size_t *lds) {
    *d_args = nullptr;
    *d_ustart = nullptr;
    std::vector<StripArgs> args(nm);
    std::vector<int64_t> ustart(nm + 1, 0);
    // one workgroup per CU with as many columns of a member as it has room
    // for: more bytes in flight than smaller workgroups with a column each
    // (12 members of 35 x 35 .. 59 x 59: 1.74 ms per launch against 1.85)
    size_t need = 0;
    for (int i = 0; i < nm; ++i) {
        const DevHam &h = *m[i].h;
        if (h.sg.s == 0 || h.n != (int64_t)h.sg.lx * h.sg.ly) return hipErrorInvalidValue;
        args[i] = strip_args(h, m[i].X, m[i].Y, m[i].ld, h.n, m[i].dts, m[i].K, m[i].reps);
        StripGeom &g = args[i].g;
        g.cols = strip_batch_cols(g);
        need = std::max(need, (size_t)g.cols * g.region * sizeof(double2));
        ustart[i + 1] = ustart[i] + (h.n + g.cols - 1) / g.cols;
    }
    StripArgs *da = nullptr;
    int64_t *du = nullptr;
    hipError_t e = lmhapi::device_malloc((void **)&da, sizeof(StripArgs) * std::max(nm, 1));
    if (e == hipSuccess) e = lmhapi::device_malloc((void **)&du, sizeof(int64_t) * (nm + 1));
    if (e == hipSuccess && nm) e = hipMemcpy(da, args.data(), sizeof(StripArgs) * nm, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(du, ustart.data(), sizeof(int64_t) * (nm + 1), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        if (da) (void)hipFree(da);
        if (du) (void)hipFree(du);
        return e;
    }
    *d_args = da;
    *d_ustart = du;
    *nunits = ustart[nm];
    *lds = need;
    return hipSuccess;
}

hipError_t launch_batched_strip(const void *d_args, const int64_t *d_ustart, int nm, int64_t nunits, size_t lds,
                                bool tout, hipStream_t st) {
    if (nunits == 0) return hipSuccess;
    static std::atomic<uint64_t> done{0};
    int cus = 0;
    hipError_t e = device_cus(&cus);
    if (e != hipSuccess) return e;
    e = once_per_device(done, [] {
        hipError_t r = hipFuncSetAttribute((const void *)batched_strip_kernel<true>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kStripLdsBytes);
        if (r == hipSuccess)
            r = hipFuncSetAttribute((const void *)batched_strip_kernel<false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kStripLdsBytes);
        return r;
    });
    if (e != hipSuccess) return e;
    const int64_t np = std::min<int64_t>(nunits, std::max(cus, 1));
    const int64_t nprog = ((np + kNumXCD - 1) / kNumXCD) * kNumXCD;
    const auto *args = static_cast<const StripArgs *>(d_args);
    if (tout)
        hipLaunchKernelGGL(batched_strip_kernel<true>, dim3((unsigned)nprog), dim3(kStripThreads), lds, st, args,
                           d_ustart, nm, nunits, nprog);
    else
        hipLaunchKernelGGL(batched_strip_kernel<false>, dim3((unsigned)nprog), dim3(kStripThreads), lds, st, args,
                           d_ustart, nm, nunits, nprog);
    return hipGetLastError();
}

hipError_t prepare_strip(const DevHam &h) {
    if (h.sg.s == 0) return hipSuccess;
    switch (strip_shape_id(h.sg.bx, h.sg.s)) {
#define LMH_STRIP_PREP(BX, S) \
    case strip_shape_id(BX, S): return h.sg.ly % S ? prepare_sx<BX, S, strip_whole(BX, S)>() : prepare_sx<BX, S, true>();
        LMH_STRIP_SHAPES(LMH_STRIP_PREP)
#undef LMH_STRIP_PREP
        default: return hipErrorInvalidValue;
    }
}

}  // namespace lmh
