// Lanczos kernels of the Krylov ket propagator (lmh_krylov_step): for every
// ket column c at once, with the basis v_j stored as (krylovdim + 1) blocks of
// ld x m complex entries and the unnormalised next vector w_j in one of two
// scratch blocks,
//     beta_j = |w_j|,  v_j = w_j / beta_j                (w_0 = psi)
//     w = H v_j - beta_j v_{j-1},  alpha_j = <v_j, w>
//     w_{j+1} = w - alpha_j v_j
// H is the context's ELL Hamiltonian (diagonal + zmax slots), applied row-wise
// with the neighbours gathered through L1/L2 (one ket column is N x 16 B; the
// matrix-free stencil is bound by the basis traffic, not by arithmetic).
// Reductions over rows go through per-block partial sums; the kernel after a
// reduction sums the partials of its column itself (nb <= a few hundred), so
// an iteration is two launches (the normalisation of w_j rides with the
// product by H) and no host round trip.  w_j is read by the neighbours of a
// row while v_j is written, hence two scratch blocks used alternately.
#include "lmhip_internal.h"

namespace lmh {

namespace {

constexpr int kLzThreads = 256;

// block sums of R values at once, in every thread, by halves: thread t adds
// those of t + 128, of t + 64, then a wavefront's by shuffles of 32 .. 1, one
// barrier in all.  The order of the sums, and which product of a complex one
// is rounded (fma below), are part of the result: alpha and beta turn the
// whole ket.  Other orders gave errors against 64-bit values of up to 6 % more
// (rms of 80 kets at N = 100352, 20 steps: 1.25 +- 0.02 and 1.32 +- 0.03 e-17).
// `red` holds kLzThreads * R doubles and is not used again before the next
// barrier.
template <int R>
__device__ __forceinline__ void block_sums(double (&v)[R], double *red) {
#pragma unroll
    for (int r = 0; r < R; ++r) red[r * kLzThreads + threadIdx.x] = v[r];
    __syncthreads();
    static_assert(kLzThreads == 256, "four wavefronts");
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const double *q = red + r * kLzThreads + lane;
        v[r] = (q[0] + q[128]) + (q[64] + q[192]);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] += __shfl_xor(v[r], off);
}

// a thread's share of a column's nb partials (fixed order)
__device__ __forceinline__ double partial_share(const double *part, int nb) {
    const int t = threadIdx.x;
    double acc = t < nb ? part[t] : 0.0;
    for (int b = t + kLzThreads; b < nb; b += kLzThreads) acc += part[b];
    return acc;
}

// v_1 = psi / |psi| for every column: partial |psi|^2 per block
__global__ void __launch_bounds__(kLzThreads) lanczos_norm_kernel(const double2 *__restrict__ X, int64_t n, int64_t ld,
                                                                 double *__restrict__ part, int nb) {
    __shared__ double red[kLzThreads];
    const int64_t c = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * kLzThreads + threadIdx.x;
    double s[1] = {0.0};
    if (i < n) {
        const double2 v = X[c * ld + i];
        s[0] = fma(v.x, v.x, v.y * v.y);
    }
    block_sums(s, red);
    if (threadIdx.x == 0) part[c * nb + blockIdx.x] = s[0];
}

// beta_j[c] = |w_j| from the column's partials of |w|^2 (one block per column).
// With ab_host the block also writes the column's alpha_0 .. alpha_{j-1} and
// beta_0 .. beta_j to the host's pinned copy: a copy after the kernel costs
// ~5 us and a gap of its own.
__global__ void __launch_bounds__(kLzThreads) lanczos_beta_kernel(const double *__restrict__ part, int nb, int64_t m, int j,
                                                                 const double *__restrict__ alpha, double *__restrict__ beta,
                                                                 double *__restrict__ alpha_host,
                                                                 double *__restrict__ beta_host) {
    __shared__ double red[kLzThreads];
    const int64_t c = blockIdx.x;
    double b[1] = {partial_share(part + c * nb, nb)};
    block_sums(b, red);
    const double bj = sqrt(b[0]);
    if (threadIdx.x == 0) beta[j * m + c] = bj;
    if (!alpha_host) return;
    for (int q = threadIdx.x; q <= j; q += kLzThreads) {
        if (q < j) alpha_host[q * m + c] = alpha[q * m + c];
        beta_host[q * m + c] = q < j ? beta[q * m + c] : bj;
    }
}

// beta_j = |W| (partials part_w); v_j = W / beta_j into Vj (0 stays 0), block 0
// recording beta_j; Wn = H v_j - beta_j v_{j-1}; partials of <v_j, Wn>.
// Bound by latency (N = 10^5: 16 MB through L2 and 392 workgroups): H W is
// formed unscaled, so its loads and gathers run while the norm is summed.
// With LDS tree sums (8 barriers each, three sums) and the loads behind the
// first of them 7.7 us, now 6.1; the kernel below 5.4, now 3.6 (N = 100352,
// 3 neighbours, one column).
// AHEAD: H's values and the previous vector are loaded in front of the sum
// too, which pays while waves are few.  With 9 slots they cost the registers
// of other waves: 100 kets at N = 20000 69 us a launch with them, 57 without
// (a step 3.22 and 3.11 ms), one ket 132 and 136 us a step.
template <int ZR, bool AHEAD>
__global__ void __launch_bounds__(kLzThreads) lanczos_matvec_kernel(
    const int32_t *__restrict__ col, const double2 *__restrict__ val, const double *__restrict__ diag, int64_t n,
    int zmax, const double2 *__restrict__ W, const double *__restrict__ part_w, double2 *__restrict__ Vj,
    const double2 *__restrict__ Vprev, double2 *__restrict__ Wn, int64_t ld, double *__restrict__ beta_out,
    double *__restrict__ part_re, double *__restrict__ part_im, int nb) {
    __shared__ double red[kLzThreads], red2[2 * kLzThreads];
    const int64_t c = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * kLzThreads + threadIdx.x;
    const bool on = i < n;
    const int64_t ic = on ? i : n - 1;
    const double2 *w = W + c * ld;
    int32_t cq[ZR];
    double2 hv[ZR];
#pragma unroll
    for (int q = 0; q < ZR; ++q) {
        cq[q] = q < zmax ? col[(int64_t)q * n + ic] : -1;
        if (AHEAD && q < zmax) hv[q] = val[(int64_t)q * n + ic];
    }
    double b[1] = {partial_share(part_w + c * nb, nb)};
    const double2 wi = w[ic];
    const double d = diag[ic];
    double2 p = make_double2(0.0, 0.0);
    if (AHEAD && Vprev) p = Vprev[c * ld + ic];
    double2 hw = make_double2(d * wi.x, d * wi.y);
#pragma unroll
    for (int q = 0; q < ZR; ++q)
        if (cq[q] >= 0) {
            const double2 h = AHEAD ? hv[q] : val[(int64_t)q * n + ic];
            const double2 x = w[cq[q]];
            hw.x += fma(h.x, x.x, -(h.y * x.y));
            hw.y += fma(h.y, x.x, h.x * x.y);
        }
    block_sums(b, red);
    if (!AHEAD && Vprev) p = Vprev[c * ld + ic];
    const double beta = sqrt(b[0]);
    const double inv = beta > 0.0 ? 1.0 / beta : 0.0;
    double dot[2] = {0.0, 0.0};                          // conj(v_i) r
    if (on) {
        const double2 vi = make_double2(wi.x * inv, wi.y * inv);
        double2 r = make_double2(hw.x * inv, hw.y * inv);       // H v_j
        if (Vprev) {
            r.x = fma(-beta, p.x, r.x);
            r.y = fma(-beta, p.y, r.y);
        }
        Vj[c * ld + i] = vi;
        Wn[c * ld + i] = r;
        dot[0] = fma(vi.y, r.y, vi.x * r.x);
        dot[1] = fma(vi.x, r.y, -(vi.y * r.x));
    }
    block_sums(dot, red2);
    if (threadIdx.x == 0) {
        part_re[c * nb + blockIdx.x] = dot[0];
        part_im[c * nb + blockIdx.x] = dot[1];
        if (blockIdx.x == 0) beta_out[c] = beta;
    }
}

// alpha = <v_j, W> from the partials; W -= alpha v_j; partials of |W|^2; block
// 0 records Re alpha
__global__ void __launch_bounds__(kLzThreads) lanczos_orth_kernel(const double2 *__restrict__ Vj, double2 *__restrict__ W,
                                                                 int64_t n, int64_t ld, const double *__restrict__ part_re,
                                                                 const double *__restrict__ part_im, int nb,
                                                                 double *__restrict__ alpha_out,
                                                                 double *__restrict__ part_nrm) {
    __shared__ double red[2 * kLzThreads], red2[kLzThreads];
    const int64_t c = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * kLzThreads + threadIdx.x;
    const int64_t ic = i < n ? i : n - 1;
    const double2 v = Vj[c * ld + ic];
    double2 w = W[c * ld + ic];
    double a[2] = {partial_share(part_re + c * nb, nb), partial_share(part_im + c * nb, nb)};
    block_sums(a, red);
    double s[1] = {0.0};
    if (i < n) {
        w.x -= fma(a[0], v.x, -(a[1] * v.y));
        w.y -= fma(a[1], v.x, a[0] * v.y);
        W[c * ld + i] = w;
        s[0] = fma(w.x, w.x, w.y * w.y);
    }
    block_sums(s, red2);
    if (threadIdx.x == 0) {
        part_nrm[c * nb + blockIdx.x] = s[0];
        if (blockIdx.x == 0) alpha_out[c] = a[0];
    }
}

// Y[:, c] = sum_{k < len[c]} coef[c][k] V_k[:, c]; len[c] < 0: a copy of X[:, c]
__global__ void __launch_bounds__(kLzThreads) krylov_combine_kernel(const double2 *__restrict__ V, int64_t vstride,
                                                                   const double2 *__restrict__ coef, int kmax,
                                                                   const int *__restrict__ len,
                                                                   const double2 *__restrict__ X, double2 *__restrict__ Y,
                                                                   int64_t n, int64_t ld) {
    const int64_t c = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * kLzThreads + threadIdx.x;
    if (i >= n) return;
    const int L = len[c];
    if (L < 0) {
        Y[c * ld + i] = X[c * ld + i];
        return;
    }
    double2 acc = make_double2(0.0, 0.0);
    for (int k = 0; k < L; ++k) {
        const double2 a = coef[c * kmax + k];
        const double2 v = V[k * vstride + c * ld + i];
        acc.x += a.x * v.x - a.y * v.y;
        acc.y += a.x * v.y + a.y * v.x;
    }
    Y[c * ld + i] = acc;
}

// the same for one ket whose coefficients fit the kernel's arguments: no
// upload in front of it (two copies of ~5 us)
struct CombineCoef {
    double2 a[kCombineArgs];
};
__global__ void __launch_bounds__(kLzThreads) krylov_combine_one_kernel(const double2 *__restrict__ V, int64_t vstride,
                                                                       CombineCoef coef, int L, double2 *__restrict__ Y,
                                                                       int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kLzThreads + threadIdx.x;
    if (i >= n) return;
    double2 acc = make_double2(0.0, 0.0);
    for (int k = 0; k < L; ++k) {
        const double2 a = coef.a[k];
        const double2 v = V[k * vstride + i];
        acc.x += a.x * v.x - a.y * v.y;
        acc.y += a.x * v.y + a.y * v.x;
    }
    Y[i] = acc;
}

}  // namespace

int lanczos_blocks(int64_t n) { return (int)((n + kLzThreads - 1) / kLzThreads); }

hipError_t launch_lanczos_start(const double2 *X, int64_t n, int64_t ld, int64_t m, double *part, hipStream_t st) {
    const int nb = lanczos_blocks(n);
    hipLaunchKernelGGL(lanczos_norm_kernel, dim3((unsigned)nb, (unsigned)m), dim3(kLzThreads), 0, st, X, n, ld, part,
                       nb);
    return hipGetLastError();
}

hipError_t launch_lanczos_iteration(const DevHam &h, const double2 *W, const double *part_w, double2 *Vj,
                                    const double2 *Vprev, double2 *Wn, int64_t ld, int64_t m, double *part_re,
                                    double *part_im, double *part_wn, double *alpha_out, double *beta_out,
                                    hipStream_t st) {
    const int64_t n = h.n;
    const int nb = lanczos_blocks(n);
    const dim3 grid((unsigned)nb, (unsigned)m);
#define LMH_LZ(ZR, AHEAD)                                                                                          \
    hipLaunchKernelGGL((lanczos_matvec_kernel<ZR, AHEAD>), grid, dim3(kLzThreads), 0, st, h.col, h.val, h.diag, n,   \
                       h.zmax, W, part_w, Vj, Vprev, Wn, ld, beta_out, part_re, part_im, nb)
    if (h.zmax <= 4)
        LMH_LZ(4, true);
    else if (h.zmax <= 9 && m <= 8)
        LMH_LZ(9, true);
    else if (h.zmax <= 9)
        LMH_LZ(9, false);
    else if (h.zmax <= 16)
        LMH_LZ(16, false);
    else
        return hipErrorInvalidValue;
#undef LMH_LZ
    hipLaunchKernelGGL(lanczos_orth_kernel, grid, dim3(kLzThreads), 0, st, Vj, Wn, n, ld, part_re, part_im, nb,
                       alpha_out, part_wn);
    return hipGetLastError();
}

hipError_t launch_lanczos_beta(const double *part, int64_t n, int64_t m, int j, const double *alpha, double *beta,
                               double *alpha_host, double *beta_host, hipStream_t st) {
    hipLaunchKernelGGL(lanczos_beta_kernel, dim3((unsigned)m), dim3(kLzThreads), 0, st, part, lanczos_blocks(n), m, j,
                       alpha, beta, alpha_host, beta_host);
    return hipGetLastError();
}

hipError_t launch_krylov_combine_one(const double2 *V, int64_t vstride, const double *coef, int len, double2 *Y,
                                     int64_t n, hipStream_t st) {
    if (len < 0 || len > kCombineArgs) return hipErrorInvalidValue;
    CombineCoef cf{};
    for (int k = 0; k < len; ++k) cf.a[k] = make_double2(coef[2 * k], coef[2 * k + 1]);
    hipLaunchKernelGGL(krylov_combine_one_kernel, dim3((unsigned)lanczos_blocks(n)), dim3(kLzThreads), 0, st, V, vstride,
                       cf, len, Y, n);
    return hipGetLastError();
}

hipError_t launch_krylov_combine(const double2 *V, int64_t vstride, const double2 *coef, int kmax, const int *len,
                                 const double2 *X, double2 *Y, int64_t n, int64_t ld, int64_t m, hipStream_t st) {
    const dim3 grid((unsigned)lanczos_blocks(n), (unsigned)m);
    hipLaunchKernelGGL(krylov_combine_kernel, grid, dim3(kLzThreads), 0, st, V, vstride, coef, kmax, len, X, Y, n,
                       ld);
    return hipGetLastError();
}

}  // namespace lmh
