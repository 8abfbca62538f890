// In-kernel Hamiltonian construction: Peierls phases from the gauge field,
// hopping amplitudes, boundary twists and on-site energies, written to an
// ELL layout that the propagation kernels read.
//
// Follows LatticeModels.jl 1.0.7:
//   src/operators/builder.jl:282-285   H[i,j] = t * twist_j * exp(-2πi ∫A·dl) * conj(twist_i)
//                                      (the angle is fl(fl(-2π) * x))
//   src/operators/builder.jl:296-309   auto-Hermitian partner H[j,i] = conj(H[i,j]);
//                                      repeated writes to one entry accumulate in order
//   src/zoo/magneticfields.jl:11-15    Landau:    (x1 + x2)(y2 - y1) B / 2
//   src/zoo/magneticfields.jl:27-31    symmetric: (x1 y2 - x2 y1) / 2 B
//   src/zoo/magneticfields.jl:72-85    axial point flux: acos(p1·p2/(|p1||p2|)/(1+1e-11))
//                                      * sign(det[p1 p2]) * flux / 2π
//   src/zoo/magneticfields.jl:89-104   singular point flux
//   src/operators/magneticfield.jl:104 field sums add left to right
// Floating-point contraction is disabled in the phase code so the operation
// order is the reference's; the bar for the phase is a few ulp.
#include "peierls.h"

#include <algorithm>

namespace lmh {

namespace {

using peierls::bond_value;

__device__ __forceinline__ double habs(double2 v) { return hypot(v.x, v.y); }

// H's entry in ELL slot q for the field components f[0 .. nf): its bonds'
// values (conjugated for the Hermitian partner) added in order
__device__ __forceinline__ double2 slot_value(const DevHam &h, int64_t q, const FieldComp *f, int64_t nf) {
    double2 acc = make_double2(0.0, 0.0);
    const int64_t c0 = h.cptr[q], c1 = h.cptr[q + 1];
    for (int64_t c = c0; c < c1; ++c) {
        const int64_t e = h.cbond[c];
        const bool partner = e < 0;
        const int64_t b = partner ? ~e : e;
        double2 v = bond_value(h, b, f, nf);
        if (partner) v.y = -v.y;
        if (c == c0) {
            acc = v;
        } else {
            acc.x += v.x;
            acc.y += v.y;
        }
    }
    return acc;
}

constexpr int kBuildLdsSlots = 64;

// H's rows, 64 to a workgroup: lane = row, thread row y = its slots y, y +
// blockDim.y, ... -- a slot's value is a chain of dependent loads and an acos
// or sincos, so the slots of a row run side by side (one thread per row, slot
// after slot, took 9-27 us for N = 100 .. 3200).  The row maxima and absolute
// sums go to one partial per workgroup (no atomics, nothing to clear
// beforehand), reduced by h_check_kernel; workgroup 0 clears its flags.
__global__ void __launch_bounds__(1024) build_h_kernel(DevHam h) {
    extern __shared__ double mag[];                 // [zmax][64] |H_ij|, for zmax <= kBuildLdsSlots
    const int lane = threadIdx.x;
    const int64_t r = blockIdx.x * (int64_t)64 + lane;
    if (blockIdx.x == 0 && lane < 2 && threadIdx.y == 0) h.red[2 + lane] = 0ull;
    if (r < h.n)
        for (int s = threadIdx.y; s < h.zmax; s += blockDim.y) {
            const int64_t q = (int64_t)s * h.n + r;
            const double2 acc = slot_value(h, q, h.field, h.nfield);
            h.val[q] = acc;
            if (h.zmax <= kBuildLdsSlots) mag[s * 64 + lane] = habs(acc);
        }
    __syncthreads();
    if (threadIdx.y != 0) return;
    double mx = 0.0, rowsum = 0.0;
    if (r < h.n) {
        const double d = h.onsite ? h.onsite[r] : 0.0;
        h.diag[r] = d;
        mx = fabs(d);
        rowsum = fabs(d);
        for (int s = 0; s < h.zmax; ++s) {
            const double a = h.zmax <= kBuildLdsSlots ? mag[s * 64 + lane] : habs(h.val[(int64_t)s * h.n + r]);
            mx = fmax(mx, a);
            rowsum += a;
        }
        if (h.rec) {
            unsigned long long cb = 0;
            for (int s = 0; s < h.zmax; ++s) {
                const int32_t c = h.col[(int64_t)s * h.n + r];
                cb |= (unsigned long long)(c < 0 ? 0 : c) << (16 * s);
            }
            h.rec[r] = make_double2(d, __longlong_as_double((long long)cb));
        }
        if (h.ndict) h.drec[r] = make_double2(d, __longlong_as_double((long long)h.dpack[r]));
    }
    for (int off = 32; off > 0; off >>= 1) {
        mx = fmax(mx, __shfl_xor(mx, off));
        rowsum = fmax(rowsum, __shfl_xor(rowsum, off));
    }
    if (lane == 0) {
        h.hpart[blockIdx.x] = mx;
        h.hpart[gridDim.x + blockIdx.x] = rowsum;
    }
}

// *flag |= bit if any lane sees bad: one atomic per wave (a field whose
// bonds all differ sets the flag from every strip)
__device__ __forceinline__ void raise_flag(unsigned long long *flag, bool bad, unsigned long long bit) {
    const unsigned long long lanes = __ballot(bad);
    if (lanes && (int)(threadIdx.x & 63) == __ffsll(lanes) - 1) atomicOr(flag, bit);
}

// After build_h, one thread per item: workgroup 0 reduces the partial maxima
// (max |H_ij| into red[0], max row sum into red[1]); the others
//   * value classes: the class table from each class's defining slot, and
//     every slot against its class (conjugated where marked) -- a difference
//     sets red[2], and the fused passes then read val instead;
//   * strips: each strip thread's bond value per direction, every used bond
//     of the strip against it bit for bit (else bit 0 of red[3]; bit 1 when an
//     x bond is complex), and the diagonal in strip order.
__global__ void __launch_bounds__(256) h_check_kernel(DevHam h, int64_t nparts) {
    if (blockIdx.x == 0) {
        __shared__ double red[2][256];
        double m[2] = {0.0, 0.0};
        for (int64_t b = threadIdx.x; b < nparts; b += 256) {
            m[0] = fmax(m[0], h.hpart[b]);
            m[1] = fmax(m[1], h.hpart[nparts + b]);
        }
        red[0][threadIdx.x] = m[0];
        red[1][threadIdx.x] = m[1];
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (threadIdx.x < w)
                for (int k = 0; k < 2; ++k) red[k][threadIdx.x] = fmax(red[k][threadIdx.x], red[k][threadIdx.x + w]);
            __syncthreads();
        }
        if (threadIdx.x < 2) h.red[threadIdx.x] = (unsigned long long)__double_as_longlong(red[threadIdx.x][0]);
        return;
    }
    const int64_t id = (blockIdx.x - 1) * (int64_t)256 + threadIdx.x;
    const int64_t n = h.n;
    if (h.ndict) {
        if (id < h.ndict) {
            const int32_t rp = h.drep[id];
            h.dval[id] = rp >= 0 ? h.val[rp] : make_double2(0.0, 0.0);
        }
        if (id < (int64_t)h.zmax * n && h.col[id] >= 0) {
            const int32_t cc = h.dcls[id];
            const int32_t rp = h.drep[cc & 0x7ff];
            double2 v = rp >= 0 ? h.val[rp] : make_double2(0.0, 0.0);
            if (cc >> 15) v.y = -v.y;
            const double2 w = h.val[id];
            raise_flag(&h.red[2], v.x != w.x || v.y != w.y, 1ull);
        }
    }
    const StripGeom &g = h.sg;
    const int S = g.s;
    if (S == 0 || id >= 5 * (int64_t)S * g.nt) return;
    // item (d, m, strip thread): d = 4 the diagonal
    const int d = (int)(id / ((int64_t)S * g.nt));
    const int rem = (int)(id - (int64_t)d * S * g.nt);
    const int m = rem / g.nt, tl = rem - m * g.nt;
    const int x = tl % g.lx, k = tl / g.lx;
    const int y0 = min(k * S, g.ly - S);
    const int64_t i0 = (int64_t)x * g.ly + y0, i = i0 + m;
    if (d == 4) {
        h.sdiag[(int64_t)m * g.nt + tl] = h.diag[i];
        return;
    }
    // the direction's first used bond of the strip (S >= 2), and this one
    bool used;
    int first = 0;
    if (d == 0) {
        used = m + 1 < S || y0 + S < g.ly || g.py;
    } else if (d == 1) {
        used = m > 0 || y0 > 0 || g.py;
        first = y0 > 0 || g.py ? 0 : 1;
    } else {
        used = d == 2 ? (x + 1 < g.lx || g.px) : (x > 0 || g.px);
    }
    const bool any = d < 2 || used;
    double2 u = make_double2(0.0, 0.0);
    bool bad = false;
    if (any) {
        const int32_t q0 = h.sslot[d * n + i0 + first];
        if (q0 >= 0) u = h.val[q0];
        if (used) {
            const int32_t q = h.sslot[d * n + i];
            if (q < 0 || q0 < 0) {
                bad = true;
            } else {
                const double2 v = h.val[q];
                bad = v.x != u.x || v.y != u.y;
                // (the kernel takes the bonds of one side of a site as the
                // conjugates of its neighbour's)
                const int32_t qc = d == 1 ? h.sslot[i0] : (d == 3 && x > 0 ? h.sslot[2 * n + i - g.ly] : -1);
                if (qc >= 0) {
                    const double2 w = h.val[qc];
                    bad = bad || v.x != w.x || v.y != -w.y;
                }
            }
        }
    }
    if (m == 0) h.stval[d * g.nt + tl] = u;
    raise_flag(&h.red[3], bad, 1ull);
    raise_flag(&h.red[3], d >= 2 && u.y != 0.0, 2ull);
}

__global__ void __launch_bounds__(256) slot_probe_kernel(DevHam h, const FieldComp *probe, int nprobe,
                                                         double2 *out) {
    const int64_t nslots = (int64_t)h.zmax * h.n;
    const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (e >= nslots * nprobe) return;
    const int64_t p = e / nslots, q = e % nslots;
    out[e] = slot_value(h, q, probe + p * h.nfield, h.nfield);
}

// Hamiltonian given as the stored values of a fixed CSC pattern: bond b takes
// nz[kup[b]] (its entry H[i_b, j_b], i_b < j_b) as its amplitude, and the
// mirrored entry nz[klo[b]] must be its exact conjugate (flag bit 0); site i
// takes the real part of its diagonal entry nz[kd[i]] (0 when not stored), whose
// imaginary part must be zero (flag bit 1); non-finite values set bit 2.
__global__ void __launch_bounds__(256) csc_gather_kernel(int64_t nbonds, int64_t n, const int64_t *__restrict__ kup,
                                                         const int64_t *__restrict__ klo,
                                                         const int64_t *__restrict__ kd,
                                                         const double2 *__restrict__ nz, double2 *__restrict__ amp,
                                                         double *__restrict__ onsite, int *__restrict__ flag) {
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t < nbonds) {
        const double2 a = nz[kup[t]], b = nz[klo[t]];
        amp[t] = a;
        if (!isfinite(a.x) || !isfinite(a.y)) atomicOr(flag, 4);
        else if (b.x != a.x || b.y != -a.y) atomicOr(flag, 1);
    } else if (t < nbonds + n) {
        const int64_t i = t - nbonds;
        const int64_t k = kd[i];
        double d = 0.0;
        if (k >= 0) {
            const double2 v = nz[k];
            d = v.x;
            if (!isfinite(v.x) || !isfinite(v.y)) atomicOr(flag, 4);
            else if (v.y != 0.0) atomicOr(flag, 2);
        }
        onsite[i] = d;
    }
}

}  // namespace

hipError_t launch_csc_gather(int64_t nbonds, int64_t n, const int64_t *kup, const int64_t *klo, const int64_t *kd,
                             const double2 *nz, double2 *amp, double *onsite, int *flag, hipStream_t st) {
    hipError_t e = hipMemsetAsync(flag, 0, sizeof(int), st);
    const int64_t work = nbonds + n;
    if (e != hipSuccess || work == 0) return e;
    hipLaunchKernelGGL(csc_gather_kernel, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, st, nbonds, n, kup, klo,
                       kd, nz, amp, onsite, flag);
    return hipGetLastError();
}

hipError_t launch_build_h(const DevHam &h, hipStream_t st) {
    if (h.n == 0) return hipSuccess;
    const int64_t nb = build_h_parts(h.n);
    const int ny = std::max(1, std::min(h.zmax, 16));
    hipLaunchKernelGGL(build_h_kernel, dim3((unsigned)nb), dim3(64, ny), h.zmax <= kBuildLdsSlots ? sizeof(double) * 64 * h.zmax : 0, st, h);
    int64_t work = h.ndict ? std::max<int64_t>((int64_t)h.zmax * h.n, h.ndict) : 0;
    if (h.sg.s > 0) work = std::max<int64_t>(work, 5 * (int64_t)h.sg.s * h.sg.nt);
    hipLaunchKernelGGL(h_check_kernel, dim3((unsigned)(1 + (work + 255) / 256)), dim3(256), 0, st, h, nb);
    return hipGetLastError();
}

hipError_t launch_slot_probe(const DevHam &h, const FieldComp *probe, int nprobe, double2 *out, hipStream_t st) {
    const int64_t work = (int64_t)h.zmax * h.n * nprobe;
    if (work == 0) return hipSuccess;
    hipLaunchKernelGGL(slot_probe_kernel, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, st, h, probe, nprobe,
                       out);
    return hipGetLastError();
}

}  // namespace lmh
