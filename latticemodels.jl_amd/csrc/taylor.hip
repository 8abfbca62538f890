// Taylor propagator for P <- U P U', U = sum_{n<=K} (-i dt H/s)^n / n!
// (applied s times per side): the reference's order rule
// (src/evolution.jl:93-118).  Column j of T_n = droptol((H/s) T_{n-1}[:, j] *
// (-i dt / n), nztol) only involves column j, so a workgroup (or a
// wavefront) walks the sites its terms reach, computes the column exactly as
// the sparse product would, drops |x| <= nztol, and notes whether any entry of
// T_n exceeds threshold/s.  K is the first n that no column exceeds: one bit
// per term and workgroup, so nothing but a 64-bit mask leaves the search.
//   * grid-stencil H: the sites within R hops, indexed directly;
//   * other H of at most 12 neighbours: a 256-site neighbourhood through an
//     LDS hash map, a thread per site with its row in registers;
//   * larger neighbourhoods: the same with 1024 and 2048 entries, a
//     wavefront per column (a table that overflows sets a flag).
// The Horner passes that apply the polynomial are in passes.hip (one term per
// launch), fused.hip, column.hip and strip.hip (all terms per launch).
#include <algorithm>

#include "lmhip_internal.h"

namespace lmh {

namespace {

// ---------------------------------------------------------------- K selection

constexpr int kWave = 64;

// lane i's value of a double, uniform i
__device__ __forceinline__ double lane_value(double v, int i) {
    union {
        double d;
        int32_t w[2];
    } u;
    u.d = v;
    u.w[0] = __builtin_amdgcn_readlane(u.w[0], i);
    u.w[1] = __builtin_amdgcn_readlane(u.w[1], i);
    return u.d;
}

// s, 1/s, threshold/s, the growth bound and the order bound from H's
// reductions (src/evolution.jl:93-104: s = nextpow(2, max|H_ij| |dt|),
// Julia's nextpow being 1 for arguments <= 1; the order bound is the first n
// with (|dt| rowsum / s)^n / n! <= threshold/s).
// A wavefront's lanes take it up together (every lane must call): lane t holds
// (|dt| rowsum / s) / (t + 1), and their products up to n are the bounds.
struct TaylorRun {
    double s, inv_s;
    double thr;                 // threshold / s
    double growth;              // |dt| rowsum / s: terms can only shrink from n + 1 > growth on
    double cn;                  // (dt / (lane + 1)) / s: term lane + 1's coefficient is -i cn
    int nmax;                   // (0: U = I)
};
__device__ TaylorRun taylor_run(const unsigned long long *red, double dt, double threshold) {
    static_assert(kMaxTaylor == kWave, "a lane per term");
    const int lane = threadIdx.x & (kWave - 1);
    const double maxabs = __longlong_as_double((long long)red[0]);
    const double rowsum = __longlong_as_double((long long)red[1]);
    TaylorRun r;
    r.s = r.inv_s = 1.0;
    r.nmax = 0;
    r.growth = 0.0;
    if (maxabs != 0.0 && dt != 0.0) {
        const double adt = fabs(dt);
        const double x = maxabs * adt;
        while (r.s < x) {
            r.s *= 2.0;
            r.inv_s *= 0.5;
        }
        r.growth = adt * rowsum * r.inv_s;
        r.nmax = kMaxTaylor;
    }
    r.thr = threshold * r.inv_s;
    r.cn = dt / (double)(lane + 1) * r.inv_s;
    double bound = r.growth / (double)(lane + 1);
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const double b = __shfl_up(bound, off);
        if (lane >= off) bound *= b;
    }
    const unsigned long long met = __ballot(bound <= r.thr);
    if (r.nmax && met) r.nmax = __ffsll(met);
    // the same in every lane: keep them in scalar registers
    r.s = lane_value(r.s, 0);
    r.inv_s = lane_value(r.inv_s, 0);
    r.thr = lane_value(r.thr, 0);
    r.growth = lane_value(r.growth, 0);
    r.nmax = __builtin_amdgcn_readfirstlane(r.nmax);
    return r;
}
// |v| > b from the square of v; the root is taken only where the squares do
// not decide (within a few roundings of b^2), and for a b whose square is not
// a normal number v is scaled first.
struct Bound {
    double b, lo, hi;
};
__device__ __forceinline__ Bound make_bound(double b) {
    const double b2 = b * b;
    const bool normal = b2 > 1e-280 && b2 < 1e280;
    return Bound{lane_value(b, 0), lane_value(normal ? b2 * (1.0 - 1e-14) : -1.0, 0),
                 lane_value(normal ? b2 * (1.0 + 1e-14) : INFINITY, 0)};
}
__device__ __forceinline__ bool exceeds_exactly(double2 v, double b) {
    if (b == 0.0) return fabs(v.x) > 0.0 || fabs(v.y) > 0.0;
    const double sc = b < 1e-140 ? 0x1p500 : (b > 1e140 ? 0x1p-500 : 1.0);
    const double x = v.x * sc, y = v.y * sc;
    return sqrt(x * x + y * y) > b * sc;
}
// T_nt's entry from the sum: scaled by -i cn, dropped when at most nztol;
// big: it exceeds thr (and was kept)
__device__ __forceinline__ double2 finish_term(double2 acc, double cn, const Bound &nz, const Bound &thr, bool &big) {
    double2 v = make_double2(acc.y * cn, -(acc.x * cn));
    const double m2 = fma(v.x, v.x, v.y * v.y);
    bool keep = m2 > nz.hi;
    big = m2 > thr.hi;
    if ((!keep && !(m2 < nz.lo)) || (!big && !(m2 < thr.lo))) {
        keep = exceeds_exactly(v, nz.b);
        big = exceeds_exactly(v, thr.b);
    }
    big = big && keep;
    if (!keep) v = make_double2(0.0, 0.0);
    return v;
}

__device__ __forceinline__ uint32_t hash_site(int32_t k, uint32_t mask) {
    return ((uint32_t)k * 2654435761u) & mask;
}

// LDS ordering among the lanes of one wavefront (no block barrier: the
// waves of a workgroup walk different columns for different numbers of terms)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void add_product(double2 &acc, double2 h, double2 t) {
    acc.x = fma(-h.y, t.y, fma(h.x, t.x, acc.x));
    acc.y = fma(h.y, t.x, fma(h.x, t.y, acc.y));
}

// a workgroup's terms above the threshold into one of kTaylorMasks words (a
// device-scope atomic on one address from every workgroup would serialise
// across the chip, ~0.1 us each), OR-ed together by taylor_finish_kernel
__device__ __forceinline__ void report_terms(unsigned long long *masks, unsigned long long mine) {
    if (mine) atomicOr(&masks[blockIdx.x % kTaylorMasks], mine);
}

// One wavefront per column, WAVES columns per workgroup, each with a
// MAXB-site neighbourhood.  A column stops after term nt once its terms can
// only shrink (growth bound |dt| rowsum / (s (nt+1)) <= 1: every entry of
// T_{nt+1} is at most that factor times max|T_nt|, and droptol only removes
// entries) and max|T_nt| <= thr: it cannot lift the maximum of any later
// term above thr, so the first n with max|T_n| <= thr is unchanged.
template <int MAXB, int WAVES>
__global__ void __launch_bounds__(kWave * WAVES) taylor_order_kernel(
    const int32_t *__restrict__ col, const double2 *__restrict__ val, const double *__restrict__ diag,
    int64_t n, int zmax, double dt, double nztol, double threshold, const unsigned long long *__restrict__ red,
    unsigned long long *__restrict__ masks, int *__restrict__ overflow) {
    const TaylorRun run = taylor_run(red, dt, threshold);
    const double growth = run.growth;
    const Bound thr = make_bound(run.thr), nz = make_bound(nztol);
    const int nmax = run.nmax;
    constexpr int HSZ = 2 * MAXB;
    constexpr uint32_t HMASK = HSZ - 1;
    __shared__ int32_t gidx_s[WAVES][MAXB];
    __shared__ double2 va_s[WAVES][MAXB];
    __shared__ double2 vb_s[WAVES][MAXB];
    __shared__ int32_t hkey_s[WAVES][HSZ];
    __shared__ int32_t hslot_s[WAVES][HSZ];
    __shared__ int32_t count_s[WAVES];
    __shared__ int32_t over_s[WAVES];
    unsigned long long above = 0;                     // bit nt-1: a column of this wave has |T_nt| > thr

    const int lane = threadIdx.x & (kWave - 1);
    const int w = threadIdx.x / kWave;
    int32_t *gidx = gidx_s[w];
    int32_t *hkey = hkey_s[w];
    int32_t *hslot = hslot_s[w];
    for (int64_t j = (int64_t)blockIdx.x * WAVES + w; j < n; j += (int64_t)gridDim.x * WAVES) {
        for (int t = lane; t < HSZ; t += kWave) hkey[t] = -1;
        wave_sync();
        if (lane == 0) {
            const uint32_t h0 = hash_site((int32_t)j, HMASK);
            hkey[h0] = (int32_t)j;
            hslot[h0] = 0;
            gidx[0] = (int32_t)j;
            va_s[w][0] = make_double2(1.0, 0.0);
            count_s[w] = 1;
            over_s[w] = 0;
        }
        wave_sync();
        int f0 = 0, f1 = 1;      // frontier: nodes added last (distance nt-1)
        double2 *cur = va_s[w], *nxt = vb_s[w];
        for (int nt = 1; nt <= nmax; ++nt) {
            // 1. add the neighbours of the frontier (distance nt)
            const int work = (f1 - f0) * zmax;
            for (int t = lane; t < work; t += kWave) {
                const int a = f0 + t / zmax;
                const int s = t - (t / zmax) * zmax;
                const int32_t k = col[(int64_t)s * n + gidx[a]];
                if (k < 0) continue;
                uint32_t hh = hash_site(k, HMASK);
                bool placed = false;
                for (int probe = 0; probe < HSZ; ++probe) {      // bounded: the table may fill
                    const int32_t old = atomicCAS(&hkey[hh], -1, k);
                    if (old == -1) {
                        const int32_t slot = atomicAdd(&count_s[w], 1);
                        if (slot < MAXB) {
                            gidx[slot] = k;
                            cur[slot] = make_double2(0.0, 0.0);
                            hslot[hh] = slot;
                        } else {
                            over_s[w] = 1;
                            hslot[hh] = -1;
                        }
                        placed = true;
                        break;
                    }
                    if (old == k) { placed = true; break; }
                    hh = (hh + 1) & HMASK;
                }
                if (!placed) over_s[w] = 1;
            }
            wave_sync();
            if (over_s[w]) break;
            const int cnt = count_s[w];
            f0 = f1;
            f1 = cnt;
            // 2. T_nt[:, j] = droptol((H T_{nt-1}) / s * (-i dt / nt))
            const double cn = lane_value(run.cn, nt - 1);
            bool big = false;
            for (int a = lane; a < cnt; a += kWave) {
                const int32_t g = gidx[a];
                const double d = diag[g];
                double2 acc = make_double2(d * cur[a].x, d * cur[a].y);
                for (int s = 0; s < zmax; ++s) {
                    const int64_t q = (int64_t)s * n + g;
                    const int32_t k = col[q];
                    if (k < 0) continue;
                    uint32_t hh = hash_site(k, HMASK);
                    int32_t sl = -1;
                    for (int probe = 0; probe < HSZ; ++probe) {
                        const int32_t kk = hkey[hh];
                        if (kk == k) { sl = hslot[hh]; break; }
                        if (kk == -1) break;
                        hh = (hh + 1) & HMASK;
                    }
                    if (sl < 0) continue;
                    const double2 hv = val[q];
                    const double2 tv = cur[sl];
                    add_product(acc, hv, tv);
                }
                bool over;
                const double2 v = finish_term(acc, cn, nz, thr, over);
                big = big || over;
                nxt[a] = v;
            }
            const bool any = __ballot(big) != 0;
            if (any) above |= 1ull << (nt - 1);
            wave_sync();
            double2 *tmp = cur;
            cur = nxt;
            nxt = tmp;
            if (!any && growth <= (double)(nt + 1)) break;     // uniform across the wave
        }
        if (over_s[w] && lane == 0) atomicExch(overflow, 1);
        wave_sync();
    }
    if (lane == 0) report_terms(masks, above);
}

// The same for a neighbourhood of at most 256 sites, a workgroup per column
// and a thread per site: site a's row (diagonal, values, the local slots of
// its neighbours) sits in thread a's registers from the level it joins, so a
// term is z LDS reads and products; every site looks its neighbours up once,
// entering those that are new.  Bound by latency (three barriers, a row load
// and a chain of LDS atomics per distance).  9 neighbours, against a wavefront
// per column with four sites per lane and a hash look-up per neighbour and
// term: 137 -> 71 us at N = 3200, 1.09 -> 0.57 ms at N = 28800.  The sums run
// over the same slots in the same order.
constexpr int kCellSites = 256;
template <int Z>
__global__ void __launch_bounds__(kCellSites) taylor_cells_kernel(
    const int32_t *__restrict__ col, const double2 *__restrict__ val, const double *__restrict__ diag, int64_t n,
    int zmax, double dt, double nztol, double threshold, const unsigned long long *__restrict__ red,
    unsigned long long *__restrict__ masks, int *__restrict__ overflow) {
    constexpr int HSZ = 2 * kCellSites;
    constexpr uint32_t HMASK = HSZ - 1;
    __shared__ int32_t gidx[kCellSites];
    __shared__ int32_t rcol[Z][kCellSites];            // a site's columns, then their hash positions (-1: none)
    __shared__ double2 vbuf[2][kCellSites + 1];        // the last slot holds 0
    __shared__ int32_t hkey[HSZ];
    __shared__ int32_t hslot[HSZ + 1];                 // (the last: an empty ELL slot's)
    __shared__ int32_t count;
    __shared__ int32_t above_s[kMaxTaylor];            // term nt has an entry above thr in this column
    const int t = threadIdx.x;
    const TaylorRun run = taylor_run(red, dt, threshold);
    const double growth = run.growth;
    const Bound thr = make_bound(run.thr), nz = make_bound(nztol);
    const int nmax = run.nmax;
    unsigned long long above = 0;
    for (int64_t j = blockIdx.x; j < n; j += gridDim.x) {
        for (int e = t; e < HSZ; e += kCellSites) hkey[e] = -1;
        if (t < kMaxTaylor) above_s[t] = 0;
        vbuf[0][t] = vbuf[1][t] = make_double2(t == 0 ? 1.0 : 0.0, 0.0);
        if (t == 0) {
            const uint32_t h0 = hash_site((int32_t)j, HMASK);
            vbuf[1][0] = vbuf[0][kCellSites] = vbuf[1][kCellSites] = make_double2(0.0, 0.0);
            hslot[HSZ] = kCellSites;
            hslot[h0] = 0;
            count = 1;
            gidx[0] = (int32_t)j;
        }
        __syncthreads();
        if (t == 0) hkey[hash_site((int32_t)j, HMASK)] = (int32_t)j;
        double d = 0.0;
        double2 hv[Z];
        int nb[Z];
#pragma unroll
        for (int q = 0; q < Z; ++q) {
            hv[q] = make_double2(0.0, 0.0);
            nb[q] = kCellSites;
        }
        int f1 = 0, f2 = 1, cur = 0;                    // [f1, f2): the sites at distance nt
        for (int nt = 0; nt <= nmax; ++nt) {
            const int front = f2 - f1;
            int cnt = f2;
            bool full = false;
            if (front > 0) {
                // 1. their rows
                if (t >= f1 && t < f2) {
                    const int32_t g = gidx[t];
                    int32_t k[Z];
#pragma unroll
                    for (int q = 0; q < Z; ++q) k[q] = q < zmax ? col[(int64_t)q * n + g] : -1;
                    d = diag[g];
#pragma unroll
                    for (int q = 0; q < Z; ++q) {
                        if (q < zmax) hv[q] = val[(int64_t)q * n + g];
                        rcol[q][t] = k[q];
                    }
#pragma unroll
                    for (int q = 0; q < Z; ++q)
                        if (k[q] < 0) hv[q] = make_double2(0.0, 0.0);
                }
                __syncthreads();
                // 2. their neighbours: where each is in the table; those not
                // seen yet join at distance nt + 1 (but none after the last
                // term).  A site that finds no room counts only if that
                // distance is reached: at distance nt it holds 0.
                const uint32_t inv = (1u << 20) / (uint32_t)front + 1;     // e / front for e < 12 front
                for (int e = t; e < front * zmax; e += kCellSites) {
                    const int q = (int)(((uint32_t)e * inv) >> 20), a = f1 + e - q * front;
                    const int32_t k = rcol[q][a];
                    int at = HSZ;
                    if (k >= 0) {
                        uint32_t hh = hash_site(k, HMASK);
                        for (int probe = 0; probe < HSZ; ++probe) {        // bounded: the table may fill
                            const int32_t old = nt < nmax ? atomicCAS(&hkey[hh], -1, k) : hkey[hh];
                            if (old == -1 && nt < nmax) {
                                const int32_t slot = atomicAdd(&count, 1);
                                if (slot < kCellSites) gidx[slot] = k;
                                hslot[hh] = min(slot, kCellSites);
                            }
                            if (old == k || old == -1) {
                                at = old == k || nt < nmax ? (int)hh : HSZ;
                                break;
                            }
                            hh = (hh + 1) & HMASK;
                        }
                    }
                    rcol[q][a] = at;
                }
                __syncthreads();
                cnt = count;
                full = cnt > kCellSites;
                if (t >= f1 && t < f2) {
#pragma unroll
                    for (int q = 0; q < Z; ++q)
                        if (q < zmax) nb[q] = hslot[rcol[q][t]];
                }
            }
            // 3. T_nt[:, j]
            if (nt > 0) {
                const double cn = lane_value(run.cn, nt - 1);
                bool big = false;
                if (t < f2) {
                    const double2 *src = vbuf[cur];
                    const double2 tc = src[t];
                    double2 acc = make_double2(d * tc.x, d * tc.y);
#pragma unroll
                    for (int q = 0; q < Z; ++q) add_product(acc, hv[q], src[nb[q]]);
                    vbuf[cur ^ 1][t] = finish_term(acc, cn, nz, thr, big);
                }
                if (__ballot(big) && (t & (kWave - 1)) == 0) above_s[nt - 1] = 1;
                cur ^= 1;
            }
            __syncthreads();
            if (nt > 0) {
                const bool any = above_s[nt - 1] != 0;
                if (any) above |= 1ull << (nt - 1);
                if (!any && growth <= (double)(nt + 1)) break;
            }
            if (full && nt < nmax) {                      // uniform
                if (t == 0) atomicExch(overflow, 1);
                break;
            }
            f1 = f2;
            f2 = cnt;
        }
        __syncthreads();
    }
    if (t == 0) report_terms(masks, above);
}

constexpr int64_t kOrderBlocks = 2048;    // persistent grid: each wave or workgroup walks several columns

template <int Z>
hipError_t launch_cells_t(const DevHam &h, double dt, double nztol, double threshold, unsigned long long *masks,
                          int *overflow, hipStream_t st) {
    hipLaunchKernelGGL(taylor_cells_kernel<Z>, dim3((unsigned)std::min<int64_t>(h.n, kOrderBlocks)), dim3(kCellSites), 0,
                       st, h.col, h.val, h.diag, h.n, h.zmax, dt, nztol, threshold, h.red, masks, overflow);
    return hipGetLastError();
}

template <int MAXB, int WAVES>
hipError_t launch_order_t(const DevHam &h, double dt, double nztol, double threshold, unsigned long long *masks,
                          int *overflow, hipStream_t st) {
    const int64_t grid = std::min<int64_t>((h.n + WAVES - 1) / WAVES, kOrderBlocks);
    hipLaunchKernelGGL((taylor_order_kernel<MAXB, WAVES>), dim3((unsigned)grid), dim3(kWave * WAVES), 0, st, h.col,
                       h.val, h.diag, h.n, h.zmax, dt, nztol, threshold, h.red, masks, overflow);
    return hipGetLastError();
}

// K = the first n <= nmax that no column exceeds threshold/s at; the
// reductions travel with it, and the step's Horner coefficients (dt / s, then
// (dt / s) / k: the divisions the host would do).  The result goes to device
// memory and straight to the host's pinned copy.  The masks and the overflow
// flag are left clear for the next search.
__global__ void __launch_bounds__(kTaylorMasks) taylor_finish_kernel(
    const unsigned long long *__restrict__ red, double dt, double threshold, unsigned long long *__restrict__ masks,
    int *__restrict__ overflow, TaylorOut *__restrict__ out, TaylorOut *__restrict__ out_host) {
    __shared__ TaylorOut o;
    static_assert(kTaylorMasks == kWave, "one wave");
    const int t = threadIdx.x;
    unsigned long long above = masks[t];
    masks[t] = 0ull;
    for (int off = kWave / 2; off > 0; off >>= 1) above |= __shfl_xor(above, off);
    const TaylorRun run = taylor_run(red, dt, threshold);
    const double dts = dt / run.s;
    if (t < 4) o.red[t] = red[t];
    if (t <= kStripMaxK) o.ck[t] = t ? dts / (double)t : 0.0;
    if (t == 0) {
        o.s = run.s;
        o.nmax = run.nmax;
        o.overflow = *overflow;
        *overflow = 0;
        o.reps = run.s <= 1073741824.0 ? (int)run.s : 0;
        o.dts = dts;
        int K = 0;
        if (run.nmax > 0) {
            const unsigned long long below = ~above & (run.nmax >= 64 ? ~0ull : (1ull << run.nmax) - 1ull);
            K = below ? __ffsll(below) : -1;
        }
        o.K = K;
    }
    __syncthreads();
    static_assert(sizeof(TaylorOut) % 8 == 0, "copied by words");
    const auto *w = reinterpret_cast<const unsigned long long *>(&o);
    for (int e = t; e < (int)(sizeof(TaylorOut) / 8); e += kWave) {
        reinterpret_cast<unsigned long long *>(out)[e] = w[e];
        reinterpret_cast<unsigned long long *>(out_host)[e] = w[e];
    }
}

// The order rule for grid-stencil H (StripGeom): T_n of column j is
// supported within n lattice hops of site j (H couples a site to itself and
// its four grid neighbours), so column j's terms live in the diamond of
// sites within Manhattan distance R of j, indexed directly instead of
// through a hash table.  The diamond is stored ring by ring (distance 0, 1,
// ..., R): the cells of term nt are the first 2 nt^2 + 2 nt + 1.  A workgroup
// takes a column, a thread a cell: its offset and the cells of its four
// neighbours are the same for every column, its row is loaded once per
// column.  A cell's sum keeps the ELL slot order; a neighbour beyond distance
// R is not stored (it holds no term: the terms computed reach distance
// nmax <= R only).  Needs nmax <= R and, along a periodic axis,
// 2 nmax + 1 <= L (the diamond must not wrap onto itself); otherwise it flags
// overflow and the hash-table kernels run.  Bound by latency (a barrier and
// an LDS round trip per term), at N = 10^4 by issue.  Against a wavefront per
// column with the cells strided over its lanes: 21 -> 8.5 us at N = 100,
// 39 -> 26 us at N = 2304 (R = 11), 55 -> 43 us at N = 10^4 (R = 9).
__device__ __forceinline__ int diamond_index(int du, int dv) {
    const int r = abs(du) + abs(dv);
    if (r == 0) return 0;
    // ring r holds 4r cells after the 2r^2 - 2r + 1 closer ones, in four
    // runs of r: (r - t, t), (-t, r - t), (t - r, -t), (t, t - r), t < r
    int seg, t;
    if (du > 0 && dv >= 0) seg = 0, t = dv;
    else if (du <= 0 && dv > 0) seg = 1, t = -du;
    else if (du < 0 && dv <= 0) seg = 2, t = -dv;
    else seg = 3, t = du;
    return 2 * r * r - 2 * r + 1 + seg * r + t;
}

__device__ __forceinline__ void diamond_cell(int a, int &du, int &dv) {
    if (a == 0) {
        du = dv = 0;
        return;
    }
    // the ring: largest r with 2r^2 - 2r + 1 <= a
    int r = (int)((1.0f + sqrtf((float)(2 * a - 1))) * 0.5f);
    while (2 * r * r - 2 * r + 1 > a) --r;
    while (2 * (r + 1) * (r + 1) - 2 * (r + 1) + 1 <= a) ++r;
    const int q = a - (2 * r * r - 2 * r + 1), seg = q / r, t = q - seg * r;
    if (seg == 0) du = r - t, dv = t;
    else if (seg == 1) du = -t, dv = r - t;
    else if (seg == 2) du = t - r, dv = -t;
    else du = t, dv = t - r;
}

template <int R, int NT>
__global__ void __launch_bounds__(NT, 6) taylor_grid_kernel(
    const uint32_t *__restrict__ sdir, const double2 *__restrict__ val, const double *__restrict__ diag, int64_t n,
    int zmax, StripGeom g, double dt, double nztol, double threshold, const unsigned long long *__restrict__ red,
    unsigned long long *__restrict__ masks, int *__restrict__ overflow) {
    constexpr int D = 2 * R * R + 2 * R + 1;          // cells within distance R
    static_assert(D <= NT, "a thread per cell");
    __shared__ double2 win[2][D + 1];                 // the last cell holds 0
    __shared__ uint16_t ncell[4][NT];
    __shared__ int32_t above_s[kMaxTaylor];           // term nt has an entry above thr in this column
    const int t = threadIdx.x;
    const TaylorRun run = taylor_run(red, dt, threshold);
    const double growth = run.growth;
    const Bound thr = make_bound(run.thr), nz = make_bound(nztol);
    const int nmax = run.nmax;
    if (!(nmax <= R && zmax <= 4 && (!g.px || 2 * nmax + 1 <= g.lx) && (!g.py || 2 * nmax + 1 <= g.ly))) {
        if (t == 0) atomicExch(overflow, 1);
        return;
    }
    // this thread's cell and its neighbours' (y + 1, y - 1, x + 1, x - 1)
    int du = 0, dv = 0;
    diamond_cell(min(t, D - 1), du, dv);
#pragma unroll
    for (int dr = 0; dr < 4; ++dr) {
        const int ndu = du + (dr == 2 ? 1 : (dr == 3 ? -1 : 0));
        const int ndv = dv + (dr == 0 ? 1 : (dr == 1 ? -1 : 0));
        ncell[dr][t] = (uint16_t)(abs(ndu) + abs(ndv) > R ? D : diamond_index(ndu, ndv));
    }
    const int reach = 2 * nmax * nmax + 2 * nmax + 1;   // cells any term of this search touches
    unsigned long long above = 0;
    const int step_x = (int)gridDim.x / g.ly, step_y = (int)gridDim.x - step_x * g.ly;
    int x0 = (int)blockIdx.x / g.ly, y0 = (int)blockIdx.x - x0 * g.ly;
    for (; x0 < g.lx; x0 += step_x, y0 += step_y) {
        if (y0 >= g.ly) {
            y0 -= g.ly;
            if (++x0 >= g.lx) break;
        }
        int xs = x0 + du, ys = y0 + dv;
        if (g.px) xs = xs < 0 ? xs + g.lx : (xs >= g.lx ? xs - g.lx : xs);
        if (g.py) ys = ys < 0 ? ys + g.ly : (ys >= g.ly ? ys - g.ly : ys);
        // a cell that is not a site stays 0
        const bool site = t < reach && xs >= 0 && xs < g.lx && ys >= 0 && ys < g.ly;
        const int64_t i = site ? (int64_t)xs * g.ly + ys : 0;
        const double d = diag[i];
        const uint32_t dirs = sdir[i];
        double2 hv[4];
        int nb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) hv[q] = val[(int64_t)(q < zmax ? q : 0) * n + i];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t dr = (dirs >> (2 * q)) & 3u;             // 0 y+, 1 y-, 2 x+, 3 x-
            nb[q] = (dirs >> (8 + q)) & 1u ? ncell[dr][t] : D;                 // empty slot: the cell that holds 0
        }
        for (int c = t; c <= D; c += NT) {
            win[0][c] = make_double2(c == 0 ? 1.0 : 0.0, 0.0);
            win[1][c] = make_double2(0.0, 0.0);
        }
        if (t < kMaxTaylor) above_s[t] = 0;
        __syncthreads();
        int cur = 0;
        for (int nt = 1; nt <= nmax + 1; ++nt) {
            // the operands of term nt are on their way while the flag of the
            // term before it decides whether this column is done
            const double2 *src = win[cur];
            const bool on = site && t < 2 * nt * nt + 2 * nt + 1;
            double2 tv[5];
            if (on) {
                tv[4] = src[t];
#pragma unroll
                for (int q = 0; q < 4; ++q) tv[q] = src[nb[q]];
            }
            if (nt > 1) {
                const bool any = above_s[nt - 2] != 0;
                if (any) above |= 1ull << (nt - 2);
                if (!any && growth <= (double)nt) break;
            }
            if (nt > nmax) break;
            const double cn = lane_value(run.cn, nt - 1);
            bool big = false;
            if (on) {
                double2 acc = make_double2(d * tv[4].x, d * tv[4].y);
#pragma unroll
                for (int q = 0; q < 4; ++q) add_product(acc, hv[q], tv[q]);
                win[cur ^ 1][t] = finish_term(acc, cn, nz, thr, big);
            }
            if (__ballot(big) && (t & (kWave - 1)) == 0) above_s[nt - 1] = 1;
            __syncthreads();
            cur ^= 1;
        }
        __syncthreads();
    }
    if (t == 0) report_terms(masks, above);
}

template <int R, int NT>
hipError_t launch_grid_t(const DevHam &h, double dt, double nztol, double threshold, unsigned long long *masks,
                         int *overflow, hipStream_t st) {
    hipLaunchKernelGGL((taylor_grid_kernel<R, NT>), dim3((unsigned)std::min<int64_t>(h.n, kOrderBlocks)), dim3(NT), 0, st,
                       h.sdir, h.val, h.diag, h.n, h.zmax, h.sg, dt, nztol, threshold, h.red, masks, overflow);
    return hipGetLastError();
}

}  // namespace

int taylor_order_levels() { return 4; }

// Grid-stencil H: level 0 the R = 9 diamond, 1 the R = 11 diamond, 2 and 3
// the hash kernel with 1024 and 2048 entries.  Other H: level 0 the 256-site
// neighbourhood, then 1024 and 2048 entries (level 3 as level 2).  A level is
// tried after the one below it overflowed (taylor_finish_kernel has cleared the
// flag and the masks).
hipError_t launch_taylor_order(const DevHam &h, double dt, double nztol, double threshold, int level,
                               unsigned long long *masks, int *overflow, hipStream_t st) {
    const bool gridh = h.sg.s > 0 && h.sdir && h.zmax > 0;
    if (gridh && level == 0) return launch_grid_t<9, 192>(h, dt, nztol, threshold, masks, overflow, st);
    if (gridh && level == 1) return launch_grid_t<11, 320>(h, dt, nztol, threshold, masks, overflow, st);
    if (!gridh && level == 0) {
        if (h.zmax <= 4) return launch_cells_t<4>(h, dt, nztol, threshold, masks, overflow, st);
        if (h.zmax <= 9) return launch_cells_t<9>(h, dt, nztol, threshold, masks, overflow, st);
        if (h.zmax <= 12) return launch_cells_t<12>(h, dt, nztol, threshold, masks, overflow, st);
        return launch_order_t<256, 4>(h, dt, nztol, threshold, masks, overflow, st);
    }
    if (level == (gridh ? 2 : 1)) return launch_order_t<1024, 1>(h, dt, nztol, threshold, masks, overflow, st);
    return launch_order_t<2048, 1>(h, dt, nztol, threshold, masks, overflow, st);
}

hipError_t launch_taylor_finish(const unsigned long long *red, double dt, double threshold, unsigned long long *masks,
                                int *overflow, TaylorOut *out, TaylorOut *out_host, hipStream_t st) {
    hipLaunchKernelGGL(taylor_finish_kernel, dim3(1), dim3(kTaylorMasks), 0, st, red, dt, threshold, masks, overflow, out,
                       out_host);
    return hipGetLastError();
}

}  // namespace lmh
