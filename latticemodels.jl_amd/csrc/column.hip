// Fused Taylor pass for any H of few neighbours: the "column" kernel.
//
// As in fused.hip a workgroup takes C whole columns of P through all K Horner
// terms on chip, thread t owning the sites t + m NT of each, but with every
// per-term stream taken out of the way:
//
//   * a thread's own y values stay in registers from term to term (the LDS
//     copy serves its neighbours only), so a site and term reads its z
//     neighbours and writes one value: 16 (z + 1) B of LDS traffic per column;
//   * H: the rows of a thread's sites stay in registers for the whole launch
//     (HREG), which a persistent workgroup loads once for all its column
//     groups; where they do not fit, a site's row is loaded while the
//     previous site is computed, slot by slot (a slot's register is refilled
//     as soon as it is used), so no load is waited for;
//   * the results leave from registers.
//
// What bounds it: the FP64 FMAs of a site (z complex products, 4 z + 4
// instructions) with the LDS reads and the write beside them.  A loop of 24
// FMAs, 4 LDS reads and a write runs at 41 clk per wave and CU on this card
// (31 for the FMAs alone); this kernel takes 52 at N = 1024 and 2304 with 4
// neighbours.  At N = 2304, K = 9 a side takes 97 us; fused.hip's kernel
// waited for H (80 B from L2 per site, term and column group, none loaded
// ahead) and took 150 us.  Streamed rows (Haldane at N = 3200, 407 us against
// 630) are bound by the L2 stream of H, 176 B per site and term over C
// columns, 14 TB/s.
//
// Reference step: src/evolution.jl:73-78; the polynomial is the reference's
// order-K Taylor polynomial (myexp!, :93-128) evaluated in Horner form.
#include <algorithm>

#include "lmhip_internal.h"

namespace lmh {

namespace {

constexpr int kColumnLdsBytes = 163840;

struct ColumnArgs {
    const int32_t *col;         // ELL, slot-major (-1: empty)
    const double2 *val;
    const double *diag;
    const uint4 *cpk;           // streamed rows: a site's columns, 16 bits each (slots 0..7)
    const uint2 *cpk2;          //                                               (slots 8..11)
    const double2 *X;
    double2 *Y;
    int64_t ld, ncols, groups, nprog;
    int n, zmax, K, reps;
    double dts;
    double ck[kStripMaxK + 1];  // dts / k for k <= kStripMaxK (a division per wave and term was a tenth of its VALU work)
};

__device__ __forceinline__ void cfma(double2 &acc, double2 h, double2 v) {
    acc.x = fma(h.x, v.x, acc.x);
    acc.x = fma(-h.y, v.y, acc.x);
    acc.y = fma(h.x, v.y, acc.y);
    acc.y = fma(h.y, v.x, acc.y);
}

// The 16-bit column of slot q (compile time) from a site's packed columns.
template <int Q>
__device__ __forceinline__ uint32_t packed_col(const uint4 &a, const uint2 &b) {
    const uint32_t w = Q < 2 ? a.x : Q < 4 ? a.y : Q < 6 ? a.z : Q < 8 ? a.w : Q < 10 ? b.x : b.y;
    return (Q & 1) ? w >> 16 : w & 0xffffu;
}

template <int Q, int N, class F>
__device__ __forceinline__ void static_for(F f) {
    if constexpr (Q < N) {
        f(std::integral_constant<int, Q>{});
        static_for<Q + 1, N>(f);
    }
}

// NT threads, SPT sites per thread, C columns per group, Z neighbour slots;
// HREG: H's rows in registers (2: and the next column's values loaded while
// one is computed; 3: and the next site's neighbours), 0: streamed; XREG: the input columns in registers (else
// re-read from X every term: reps == 1 only); W: waves per SIMD.
template <int NT, int SPT, int C, int Z, int HREG, bool XREG, int W, bool TOUT>
__global__ void __launch_bounds__(NT, W) column_kernel(ColumnArgs a) {
    extern __shared__ double2 lds[];             // [C][LS]
    const int t = threadIdx.x;
    const int n = a.n, zmax = a.zmax;
    const int LS = n;
    // rows in registers: one column in two LDS copies used in turn, one
    // barrier per term (a copy is written again after the barrier that
    // follows its readers' term), and the next column's values are loaded
    // while this one is computed
    constexpr bool DB = HREG;
    static_assert(!HREG || (C == 1 && XREG), "rows in registers: one column, x in registers");
    const int wbase = __builtin_amdgcn_readfirstlane(t & ~63);
    // a wave without sites among its m-th ones skips them (uniform)
    auto wave_live = [&](int m) { return m * NT + wbase < n; };
    auto site = [&](int m) { return min(t + m * NT, n - 1); };

    constexpr int HS = HREG ? SPT : 1, HZ = HREG ? Z : 1;
    constexpr bool PACK = SPT > 4;               // two 16-bit LDS byte offsets to a register (n <= 4096)
    static_assert(!HREG || !PACK || NT * SPT <= 4096, "packed offsets");
    constexpr int HC = HREG ? (PACK ? (Z + 1) / 2 : Z) : 1;
    double2 hv[HS][HZ];
    uint32_t hc[HS][HC];
    double hd[HS];
    if constexpr (HREG) {
#pragma unroll
        for (int m = 0; m < SPT; ++m) {
            const int s = site(m);
            hd[m] = a.diag[s];
            uint32_t c[Z + 1];
#pragma unroll
            for (int q = 0; q < Z; ++q) {
                const int32_t cq = q < zmax ? a.col[(int64_t)q * n + s] : -1;
                c[q] = (cq < 0 ? s : cq) * 16;   // LDS byte offset; empty slot: the site itself, value 0
                hv[m][q] = cq < 0 ? make_double2(0.0, 0.0) : a.val[(int64_t)q * n + s];
            }
            c[Z] = 0;
            if constexpr (PACK) {
#pragma unroll
                for (int q = 0; q < HC; ++q) hc[m][q] = c[2 * q] | c[2 * q + 1] << 16;
            } else {
#pragma unroll
                for (int q = 0; q < Z; ++q) hc[m][q] = c[q];
            }
        }
    }

    // consecutive groups on one XCD: the conjugate-transposed stores of
    // neighbouring columns meet in one L2
    const int64_t per = a.nprog / kNumXCD;
    const int64_t g0 = (blockIdx.x % kNumXCD) * per + blockIdx.x / kNumXCD;
    constexpr bool PF = HREG >= 2, PIPE = HREG >= 3;
    double2 xn1[PF ? SPT : 1];
    auto load_next = [&](int64_t j) {
        if constexpr (PF) {
#pragma unroll
            for (int m = 0; m < SPT; ++m) xn1[m] = a.X[min(j, a.ncols - 1) * a.ld + site(m)];
        }
    };
    load_next(g0);
    for (int64_t g = g0; g < a.groups; g += a.nprog) {
        const int64_t jb = g * C;
        double2 yr[SPT][C];
        double2 xr[XREG ? SPT : 1][XREG ? C : 1];
#pragma unroll
        for (int m = 0; m < SPT; ++m)
#pragma unroll
            for (int cc = 0; cc < C; ++cc) {
                const bool live = t + m * NT < n && jb + cc < a.ncols;
                if constexpr (PF)
                    yr[m][cc] = xn1[m];
                else
                    yr[m][cc] = live ? a.X[(jb + cc) * a.ld + t + m * NT] : make_double2(0.0, 0.0);
                if constexpr (XREG) xr[m][cc] = yr[m][cc];
            }
        load_next(jb + a.nprog);
        if constexpr (DB) {
#pragma unroll
            for (int m = 0; m < SPT; ++m)
                if (t + m * NT < n) lds[t + m * NT] = yr[m][0];
            __syncthreads();
        }
        for (int r = 0; r < a.reps; ++r) {
            if constexpr (DB) {
                // one term: neighbours from LDS copy BUF, each new value to
                // the other copy as it is made (a write costs as much LDS
                // time as three reads, 75 against 216 B/clk, and is hidden
                // behind the sites that follow)
                auto term = [&](int k, auto bufc) {
                    constexpr int BUF = decltype(bufc)::value;
                    const char *src = reinterpret_cast<const char *>(lds) + BUF * NT * SPT * 16;
                    char *dst = reinterpret_cast<char *>(lds) + (BUF ^ 1) * NT * SPT * 16;
                    const double ck = k <= kStripMaxK ? a.ck[k] : a.dts / (double)k;
                    double2 gv[PIPE ? 2 : 1][Z];
                    auto gather = [&](int m, double2 *v) {
#pragma unroll
                        for (int q = 0; q < Z; ++q) {
                            const uint32_t c = PACK ? ((q & 1) ? hc[m][q / 2] >> 16 : hc[m][q / 2] & 0xffffu) : hc[m][q];
                            v[q] = *reinterpret_cast<const double2 *>(src + c);
                        }
                    };
                    if (PIPE && wave_live(0)) gather(0, gv[0]);
                    static_for<0, SPT>([&](auto mc) {
                        constexpr int m = decltype(mc)::value;
                        if (wave_live(m)) {
                            if constexpr (!PIPE) {
                                gather(m, gv[0]);
                            } else if constexpr (m + 1 < SPT) {
                                if (wave_live(m + 1)) gather(m + 1, gv[(m + 1) & 1]);
                                __builtin_amdgcn_sched_barrier(0);
                            }
                            const double2 y = yr[m][0];
                            double2 acc = make_double2(hd[m] * y.x, hd[m] * y.y);
#pragma unroll
                            for (int q = 0; q < Z; ++q) cfma(acc, hv[m][q], gv[PIPE ? m & 1 : 0][q]);
                            yr[m][0] = make_double2(fma(ck, acc.y, xr[m][0].x), fma(-ck, acc.x, xr[m][0].y));
                            if (t + m * NT < n) *reinterpret_cast<double2 *>(dst + (t + m * NT) * 16) = yr[m][0];
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    });
                    __syncthreads();
                };
                int k = a.K;
                for (; k >= 2; k -= 2) {
                    term(k, std::integral_constant<int, 0>{});
                    term(k - 1, std::integral_constant<int, 1>{});
                }
                if (k == 1) {
                    term(1, std::integral_constant<int, 0>{});
                    // another repetition starts from copy 0
                    if (r + 1 < a.reps) {
#pragma unroll
                        for (int m = 0; m < SPT; ++m)
                            if (t + m * NT < n) lds[t + m * NT] = yr[m][0];
                        __syncthreads();
                    }
                }
            } else {
                for (int k = a.K; k >= 1; --k) {
                    const double ck = k <= kStripMaxK ? a.ck[k] : a.dts / (double)k;
                    // opaque copies: keep the per-site addresses of the
                    // streamed rows and of x from being hoisted out of the
                    // term loop
                    int nn = n;
                    int64_t ldo = a.ld;
                    asm volatile("" : "+s"(nn), "+s"(ldo));
                    // a row in flight: the next site's slots are loaded as
                    // this one's are used
                    double2 rv[Z];
                    uint4 ca = make_uint4(0, 0, 0, 0);
                    uint2 cb = make_uint2(0, 0);
                    double d;
                    double2 xn[C];
                    auto load_x = [&](int m) {
                        if constexpr (!XREG) {
                            const int s = min(t + m * NT, nn - 1);
#pragma unroll
                            for (int cc = 0; cc < C; ++cc) xn[cc] = a.X[min(jb + cc, a.ncols - 1) * ldo + s];
                        }
                    };
                    {
                        const int s = min(t, nn - 1);
                        ca = a.cpk[s];
                        if constexpr (Z > 8) cb = a.cpk2[s];
                        d = a.diag[s];
#pragma unroll
                        for (int q = 0; q < Z; ++q) rv[q] = q < zmax ? a.val[(uint32_t)(q * nn + s)] : make_double2(0.0, 0.0);
                        load_x(0);
                    }
                    // (the first row is on its way) the previous term's reads are
                    // done; publish this term's input
                    __syncthreads();
#pragma unroll
                    for (int m = 0; m < SPT; ++m)
                        if (t + m * NT < n) {
#pragma unroll
                            for (int cc = 0; cc < C; ++cc) lds[cc * LS + t + m * NT] = yr[m][cc];
                        }
                    __syncthreads();
#pragma unroll
                    for (int m = 0; m < SPT; ++m) {
                        if (!wave_live(m)) continue;
                        const int sn = min(t + (m + 1) * NT, nn - 1);
                        const bool more = m + 1 < SPT;
                        double2 acc[C];
#pragma unroll
                        for (int cc = 0; cc < C; ++cc) acc[cc] = make_double2(d * yr[m][cc].x, d * yr[m][cc].y);
                        if (more) d = a.diag[sn];
                        const uint4 cu = ca;
                        const uint2 cv = cb;
                        if (more) {
                            ca = a.cpk[sn];
                            if constexpr (Z > 8) cb = a.cpk2[sn];
                        }
                        static_for<0, Z>([&](auto qc) {
                            constexpr int q = decltype(qc)::value;
                            const uint32_t c = packed_col<q>(cu, cv);
                            if (q < zmax) {
#pragma unroll
                                for (int cc = 0; cc < C; ++cc) cfma(acc[cc], rv[q], lds[cc * LS + c]);
                                if (more) rv[q] = a.val[(uint32_t)(q * nn + sn)];
                            }
                            if constexpr (q % 3 == 2) __builtin_amdgcn_sched_barrier(0);
                        });
#pragma unroll
                        for (int cc = 0; cc < C; ++cc) {
                            const double2 x = XREG ? xr[XREG ? m : 0][XREG ? cc : 0] : xn[cc];
                            yr[m][cc] = make_double2(fma(ck, acc[cc].y, x.x), fma(-ck, acc[cc].x, x.y));
                        }
                        if (more) load_x(m + 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            if constexpr (XREG) {
                if (r + 1 < a.reps) {
#pragma unroll
                    for (int m = 0; m < SPT; ++m)
#pragma unroll
                        for (int cc = 0; cc < C; ++cc) xr[m][cc] = yr[m][cc];
                }
            }
        }
        // the next column's values are taken here: a wait for them after the
        // stores below would wait for the stores too (one in-order counter)
        if constexpr (PF) {
#pragma unroll
            for (int m = 0; m < SPT; ++m) asm volatile("" : "+v"(xn1[m].x), "+v"(xn1[m].y));
        }
        // a site's C results: one run of a row of Y (conjugate-transposed)
        // or one value in each of its columns
        int64_t ldo = a.ld;
        asm volatile("" : "+s"(ldo));
        double2 *yo = TOUT ? a.Y + t * ldo + jb : a.Y + jb * ldo + t;
#pragma unroll
        for (int m = 0; m < SPT; ++m) {
            if (t + m * NT < n) {
#pragma unroll
                for (int cc = 0; cc < C; ++cc) {
                    if (jb + cc >= a.ncols) continue;
                    if constexpr (TOUT)
                        yo[cc] = make_double2(yr[m][cc].x, -yr[m][cc].y);
                    else
                        yo[cc * ldo] = yr[m][cc];
                }
            }
            yo += TOUT ? NT * ldo : NT;
        }
    }
}

// {threads, sites per thread, columns, slots, H in registers, x in registers, waves per SIMD}
#define LMH_COLUMN_CASES(X)                                                                                       \
    X(0, 128, 1, 1, 4, 3, true, 4) X(1, 256, 1, 1, 4, 3, true, 4) X(2, 256, 2, 1, 4, 3, true, 4)                   \
    X(3, 256, 4, 1, 4, 2, true, 3) X(4, 512, 2, 1, 4, 3, true, 4) X(5, 512, 3, 1, 4, 3, true, 2)                   \
    X(6, 1024, 2, 1, 4, 3, true, 4) X(7, 512, 4, 1, 4, 3, true, 2) X(8, 768, 3, 1, 4, 3, true, 3)                  \
    X(9, 512, 5, 1, 4, 3, true, 2) X(10, 768, 4, 1, 4, 2, true, 3) X(11, 768, 5, 1, 4, 1, true, 3)                 \
    X(12, 512, 8, 1, 4, 1, true, 2) X(13, 256, 1, 1, 9, 3, true, 4) X(14, 512, 2, 1, 9, 1, true, 4)                \
    X(15, 512, 4, 1, 9, 1, true, 2) X(16, 512, 5, 3, 9, 0, false, 2) X(17, 512, 7, 3, 9, 0, false, 2)              \
    X(18, 512, 7, 2, 9, 0, true, 2) X(19, 512, 10, 2, 9, 0, false, 2) X(20, 512, 20, 1, 9, 0, true, 2)
constexpr size_t column_lds(int c, bool hreg, int64_t stride) {
    return std::min<size_t>((size_t)(hreg && c == 1 ? 2 : c) * stride * sizeof(double2), kColumnLdsBytes);
}

struct ColumnVariant {
    int nt, spt, c, z;
    int hreg;
    bool xreg;
    int w;
};
#define LMH_COLUMN_ROW(idx, nt, spt, c, z, hreg, xreg, w) {nt, spt, c, z, hreg, xreg, w},
constexpr ColumnVariant kColumnVariants[] = {LMH_COLUMN_CASES(LMH_COLUMN_ROW)};
#undef LMH_COLUMN_ROW
constexpr int kNumColumnVariants = sizeof(kColumnVariants) / sizeof(kColumnVariants[0]);

template <int NT, int SPT, int C, int Z, int HREG, bool XREG, int W, bool TOUT>
hipError_t launch_column_t(const ColumnArgs &a, hipStream_t st) {
    const size_t lds = column_lds(C, HREG, HREG ? NT * SPT : a.n);
    static std::atomic<uint64_t> done{0};
    static std::atomic<int> resident{0};     // workgroups at once (streamed rows: at the largest n)
    hipError_t e = once_per_device(done, [] {
        hipError_t r = hipFuncSetAttribute((const void *)column_kernel<NT, SPT, C, Z, HREG, XREG, W, TOUT>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kColumnLdsBytes);
        int per_cu = 0, dev = 0, cus = 0;
        if (r == hipSuccess)
            r = hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, (const void *)column_kernel<NT, SPT, C, Z, HREG, XREG, W, TOUT>, NT,
                column_lds(C, HREG, NT * SPT));
        if (r == hipSuccess) r = hipGetDevice(&dev);
        if (r == hipSuccess) r = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (r == hipSuccess) resident.store(std::max(1, per_cu) * std::max(1, cus));
        return r;
    });
    if (e != hipSuccess || a.ncols == 0) return e;
    ColumnArgs b = a;
    b.groups = (a.ncols + C - 1) / C;
    const int64_t np = std::min<int64_t>(b.groups, resident.load());
    b.nprog = (np + kNumXCD - 1) / kNumXCD * kNumXCD;
    hipLaunchKernelGGL((column_kernel<NT, SPT, C, Z, HREG, XREG, W, TOUT>), dim3((unsigned)b.nprog), dim3(NT), lds, st,
                       b);
    return hipGetLastError();
}

template <bool TOUT>
hipError_t dispatch_column(int v, const ColumnArgs &a, hipStream_t st) {
    switch (v) {
#define LMH_COLUMN_CASE(idx, nt, spt, c, z, hreg, xreg, w) \
    case idx: return launch_column_t<nt, spt, c, z, hreg, xreg, w, TOUT>(a, st);
        LMH_COLUMN_CASES(LMH_COLUMN_CASE)
#undef LMH_COLUMN_CASE
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

int column_variant_count() { return kNumColumnVariants; }

bool column_variant_valid(int v, int64_t n, int zmax) {
    if (v < 0 || v >= kNumColumnVariants) return false;
    const ColumnVariant &w = kColumnVariants[v];
    return n > 0 && n <= (int64_t)w.nt * w.spt && w.c * n * 16 <= kColumnLdsBytes && zmax <= w.z;
}

// Rows of at most 4 slots: in registers up to n = 4096, where a column is
// split over enough threads that they fit (timed on open squares in a point
// flux, K = 9, us per pass, against the general kernel by size: N = 100 6.4 /
// 10.3, 484 10.9 / 14.9, 1024 25 / 33, 1936 74 / 95, 2304 97 / 150, 2916
// 177 / 222, 3600 288 / 474, 4096 428 / 522); above, H must be streamed and
// the general kernel's 80 B per site are the smaller stream.  Up to 9 slots
// in registers up to n = 2048 (Haldane, K = 6: N = 512 18 / 51, 1984
// 106 / 146), streamed above, where the threads' number of rows decides (us
// per step, K = 7 .. 8, streamed / general): 5 slots N = 2450 361 / 459, 2888
// 538 / 564, 3528 696 / 1048, 3872 1078 / 1212, 4232 1458 / 1403, 5000 1871 /
// 1668; 6 slots 2601 520 / 479, 3481 759 / 1047, 3969 1195 / 1238, 4356 1617 /
// 1428; 8 slots 2500 498 / 530, 2601 668 / 542, 3136 920 / 1115, 3600 1352 /
// 1318, 4096 1597 / 1407, 5041 2401 / 1911; 9 slots 2450 467 / 613, 2592 644 /
// 634, 2888 713 / 673, 3528 942 / 1373, 4232 1794 / 1823, 5000 2233 / 2184.
// So from 6 slots on a sixth row of 512 threads goes to the general kernel
// (which has 1024 with three each), except that with 9 a wave's worth of it
// costs nothing; rows past the seventh with 7 or 8 slots, past the eighth with
// 5 or 6 (with 9 the general kernel loads 12 slots and both are within 2 %).
// Few columns (at most two to a CU) are one round of either, and the streamed
// rows the shorter one up to more of them (48 kets: 5 slots N = 3698 50 / 66;
// 7 slots 3698 69 / 73; 8 slots 2704 55 / 59, 3600 74 / 74, 4096 80 / 75;
// 9 slots 2592 52 / 70, 4608 84 / 87).
// Above n = 5120 one column fills the LDS and the streamed rows win again
// (8 slots 5184 3365 / 5163, 10201 11248 / 11602; 9 slots 10082 10735 / 14073).
int column_default_variant(int64_t n, int zmax, int64_t ncols) {
    if (zmax <= 4) {
        if (n > 4096) return -1;
        return n <= 128 ? 0 : n <= 256 ? 1 : n <= 512 ? 2 : n <= 1024 ? 4 : n <= 2048 ? 6 : n <= 2304 ? 8
               : n <= 3072 ? 10 : n <= 3840 ? 11 : 12;
    }
    if (zmax > 9 || n > 10240) return -1;
    const bool few = ncols <= 512;
    if (n <= 2560) return n <= 256 ? 13 : n <= 2048 ? 15 : 16;
    if (n <= 3072 && zmax > 5 && !few) return zmax == 9 && n <= 2560 + 64 ? 17 : -1;
    if (n <= 3584) return 18;
    if (n <= 5120) {
        const int64_t last = zmax == 9 ? 5120 : zmax == 8 ? 3584 : zmax == 7 ? (few ? 4096 : 3584) : (few ? 5120 : 4096);
        return n <= last ? 19 : -1;
    }
    return 20;
}

bool column_variant_runs(int v, const DevHam &h, int reps) {
    return column_variant_valid(v, h.n, h.zmax) && (kColumnVariants[v].hreg || h.cpk) &&
           (kColumnVariants[v].xreg || reps == 1);
}

hipError_t launch_column(int v, const DevHam &h, const double2 *X, double2 *Y, int64_t ld, int64_t ncols,
                         double dt_over_s, int K, int reps, bool tout, hipStream_t st) {
    if (!column_variant_runs(v, h, reps) || (tout && ncols != h.n)) return hipErrorInvalidValue;
    ColumnArgs a{h.col, h.val, h.diag, h.cpk, h.cpk2, X, Y, ld, ncols, 0, 0, (int)h.n, h.zmax, K, reps, dt_over_s, {}};
    for (int k = 1; k <= kStripMaxK; ++k) a.ck[k] = dt_over_s / (double)k;
    return tout ? dispatch_column<true>(v, a, st) : dispatch_column<false>(v, a, st);
}

}  // namespace lmh
