// C ABI, setup (hierarchy build) and the PCG driver of the MI355X pressure
// Poisson solver. Replaces hypre_str with method pcg_pfmg
// (src/solver/hypre_str_class.f90:264-284 in the NGA2 tree).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <type_traits>
#include <vector>

#include "ngap_internal.h"
#include "ngapsolve.h"
#include "ngapsolve_test.h"

using namespace ngap;

namespace {

// ---------------------------------------------------------------- scalar slots
enum { S_RR = 0, S_BB, S_RHO, S_ALPHA, S_BETA, S_PQ, S_RHO0, S_BAD, S_RRT, S_ASYM, S_STR0, S_STR1, S_STR2, S_CSING,
       S_CBAD, S_XNZ, S_NSCAL };
constexpr int NSCAL_ALLOC = 16;
// device and pinned host scalars, then 4 int flags in the same allocation
constexpr size_t SCAL_BYTES = sizeof(double) * NSCAL_ALLOC + sizeof(int) * 4;

struct Ghost {
    long long nxo, nyo;
    int oi, oj, ok;
};

struct Slots {
    int s[7];  // stencil slot of centre, +x, -x, +y, -y, +z, -z
    int nst;
};

__device__ __forceinline__ long long gidx(const Ghost &h, int i, int j, int k) {
    return (long long)(i + h.oi) + h.nxo * ((long long)(j + h.oj) + h.nyo * (long long)(k + h.ok));
}

// cell coordinates of p < 2^31 (setup rejects larger grids), in 32 bits
__device__ __forceinline__ void decomp0(const Geo &g, long long p, int &i, int &j, int &k) {
    const unsigned q = (unsigned)p, r = q / (unsigned)g.n0;
    i = (int)(q - r * (unsigned)g.n0);
    k = (int)(r / (unsigned)g.n1);
    j = (int)(r - (unsigned)k * (unsigned)g.n1);
}

// ---------------------------------------------------------------- setup kernels

// Level-0 symmetric storage from the ghosted AoS opr (hypre_str_class.f90:
// 171-179: rows with opr(1)==0 become identity rows).
//
// The 7 entries of a cell are adjacent in opr, so a block's consecutive cells
// own one contiguous run per grid row. The block first copies its cells'
// entries through LDS with coalesced 8-byte loads (and, with opr_copy, writes
// them to the solver's own copy in the same coalesced order); each thread then
// takes its cell's entries from LDS. The minus neighbours' centre and plus
// coupling are read from memory.
constexpr int OPR_NST = 7;  // init accepts 7-point stencils only
__global__ void __launch_bounds__(NT) k_level0(Geo g, Ghost gh, Slots sl, const double *__restrict__ opr,
                                               double *__restrict__ opr_copy, double *__restrict__ c,
                                               double *__restrict__ a0, double *__restrict__ a1,
                                               double *__restrict__ a2, LevelData<float> s32,
                                               unsigned char *__restrict__ part, double *__restrict__ p_asym,
                                               double *__restrict__ p_bad) {
    __shared__ double sm[NT / 64];
    __shared__ double st[NT * OPR_NST];
    __shared__ int sg[NT];
    double asym = 0.0, bad = 0.0;
    const int n3[3] = {g.n0, g.n1, g.n2}, per3[3] = {g.p0, g.p1, g.p2};
    // cell indices fit in int (setup rejects 2^31 cells); the loop counter is
    // 64-bit so that its last step past N cannot overflow. The loop is uniform
    // over the block (barriers inside).
    for (long long pb = (long long)blockIdx.x * NT; pb < g.N; pb += (long long)gridDim.x * NT) {
        const bool ok = pb + threadIdx.x < g.N;
        const int p = ok ? (int)(pb + threadIdx.x) : 0;
        int c3[3] = {0, 0, 0};
        if (ok) {
            const unsigned rq = (unsigned)p / (unsigned)g.n0;
            c3[0] = p - (int)rq * g.n0;
            c3[1] = (int)(rq % (unsigned)g.n1);
            c3[2] = (int)(rq / (unsigned)g.n1);
        }
        __syncthreads();  // the previous cells' entries are no longer read
        sg[threadIdx.x] = ok ? (int)gidx(gh, c3[0], c3[1], c3[2]) : -1;
        __syncthreads();
        for (int e = threadIdx.x; e < NT * OPR_NST; e += NT) {
            const int cl = e / OPR_NST, q = e - cl * OPR_NST;
            const int gs = sg[cl];
            if (gs >= 0) {
                const double val = opr[(long long)gs * OPR_NST + q];
                st[e] = val;
                if (opr_copy) opr_copy[(long long)gs * OPR_NST + q] = val;
            }
        }
        __syncthreads();
        if (!ok) continue;
        double v[7];
        for (int s = 0; s < 7; s++) {
            v[s] = st[threadIdx.x * OPR_NST + sl.s[s]];
            if (!isfinite(v[s])) bad += 1.0;
        }
        const bool pt = fabs(v[0]) > 0.0;
        part[p] = pt ? 1 : 0;
        double cc = pt ? v[0] : 1.0;
        double av[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            av[d] = 0.0;
            double am = v[2 + 2 * d], ap = v[1 + 2 * d];
            if (n3[d] == 1) {
                if (per3[d] && pt) cc += am + ap;
                continue;
            }
            int q = nbm(c3[d], n3[d], per3[d]);
            if (q < 0 || !pt) continue;
            int e3[3] = {c3[0], c3[1], c3[2]};
            e3[d] = q;
            const double *B = opr + gidx(gh, e3[0], e3[1], e3[2]) * OPR_NST;
            if (!(fabs(B[sl.s[0]]) > 0.0)) continue;
            double apn = B[sl.s[1 + 2 * d]];
            av[d] = 0.5 * (am + apn);
            double rel = fabs(am - apn) / fabs(v[0]);
            if (rel > asym) asym = rel;
        }
        c[p] = cc;
        a0[p] = av[0];
        a1[p] = av[1];
        a2[p] = av[2];
        if (s32.c) {
            s32.c[p] = (float)cc;
            s32.a0[p] = (float)av[0];
            s32.a1[p] = (float)av[1];
            s32.a2[p] = (float)av[2];
        }
    }
    double m = block_max(asym, sm);
    double b = block_sum(bad, sm);
    if (threadIdx.x == 0) {
        p_asym[blockIdx.x] = m;
        p_bad[blockIdx.x] = b;
    }
}

// ---------------------------------------------------------------- solve kernels

// dst = part ? src(ghosted) : 0; counts non-finite values of participating
// cells (p_bad) and values that are not zero (p_nz)
__global__ void __launch_bounds__(NT) k_gather(Geo g, Ghost gh, const double *__restrict__ src,
                                               const unsigned char *__restrict__ part, double *__restrict__ dst,
                                               double *__restrict__ p_bad, double *__restrict__ p_nz) {
    __shared__ double sm[NT / 64];
    double bad = 0.0, nz = 0.0;
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < g.N; p += (long long)gridDim.x * NT) {
        int i, j, k;
        decomp0(g, p, i, j, k);
        double v = part[p] ? src[gidx(gh, i, j, k)] : 0.0;
        if (!isfinite(v)) bad += 1.0;
        if (v != 0.0) nz += 1.0;
        dst[p] = v;
    }
    if (p_bad) {
        double b = block_sum(bad, sm);
        if (threadIdx.x == 0) p_bad[blockIdx.x] = b;
    }
    if (p_nz) {
        double b = block_sum(nz, sm);
        if (threadIdx.x == 0) p_nz[blockIdx.x] = b;
    }
}

__global__ void __launch_bounds__(NT) k_scatter(Geo g, Ghost gh, const double *__restrict__ src,
                                                double *__restrict__ dst) {
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < g.N; p += (long long)gridDim.x * NT) {
        int i, j, k;
        decomp0(g, p, i, j, k);
        dst[gidx(gh, i, j, k)] = src[p];
    }
}

// The six neighbours of a cell: flat offsets, 0 where there is none (has bit q)
struct Nb6 {
    int o[6];
    int has;
};
__device__ __forceinline__ Nb6 nb6(const Geo &g, int i, int j, int k) {
    const int plane = g.n0 * g.n1;
    const int ip = nbp(i, g.n0, g.p0), im = nbm(i, g.n0, g.p0);
    const int jp = nbp(j, g.n1, g.p1), jm = nbm(j, g.n1, g.p1);
    const int kp = nbp(k, g.n2, g.p2), km = nbm(k, g.n2, g.p2);
    Nb6 n;
    n.o[0] = ip >= 0 ? ip - i : 0;
    n.o[1] = im >= 0 ? im - i : 0;
    n.o[2] = jp >= 0 ? (jp - j) * g.n0 : 0;
    n.o[3] = jm >= 0 ? (jm - j) * g.n0 : 0;
    n.o[4] = kp >= 0 ? (kp - k) * plane : 0;
    n.o[5] = km >= 0 ? (km - k) * plane : 0;
    n.has = (ip >= 0) | (im >= 0) << 1 | (jp >= 0) << 2 | (jm >= 0) << 3 | (kp >= 0) << 4 | (km >= 0) << 5;
    return n;
}

// The two exact products below are bound by the latency of their loads: a
// thread works on PU cells of its stride at a time, all loads issued before
// the first use and none behind a branch.
constexpr int PU = 2;

// r = b - A x with the exact 7-array operator (identity rows where the
// centre is 0; couplings out of a non-periodic box ignored); partial ||r||^2.
// The 7 entries of a cell are adjacent in opr, 56 bytes from cell to cell, so a
// wave copies the entries of its 64 consecutive cells through LDS with
// coalesced 8-byte loads. 256^3: 444 us one cell at a time, each lane reading
// its own entries; 309 us now.
__global__ void __launch_bounds__(NT) k_exact_resid(Geo g, Ghost gh, Slots sl, const double *__restrict__ opr,
                                                    const double *__restrict__ b, const double *__restrict__ x,
                                                    double *__restrict__ r, double *__restrict__ part) {
    __shared__ double sm[NT / 64];
    __shared__ double st[PU * NT * OPR_NST];
    double *w = st + (threadIdx.x & ~63u) * (PU * OPR_NST);  // this wave's entries
    const int lane = threadIdx.x & 63;
    const long long stride = (long long)gridDim.x * NT;
    double acc = 0.0;
    for (long long pw = blockIdx.x * (long long)NT + (threadIdx.x & ~63u); pw < g.N; pw += PU * stride) {
        int p[PU];
        Nb6 nb[PU];
        double av[PU][OPR_NST], xv[PU][7], bv[PU];
#pragma unroll
        for (int u = 0; u < PU; u++) {
            const long long q = pw + u * stride + lane;
            p[u] = q < g.N ? (int)q : (int)g.N - 1;
            int i, j, k;
            decomp0(g, p[u], i, j, k);
            const int gs = (int)gidx(gh, i, j, k);  // ghosted cells fit in 31 bits (checked at setup)
#pragma unroll
            for (int m = 0; m < OPR_NST; m++) {
                const int e = lane + 64 * m, cl = e / OPR_NST, c = e - cl * OPR_NST;
                av[u][m] = opr[(long long)__shfl(gs, cl, 64) * OPR_NST + c];
            }
            nb[u] = nb6(g, i, j, k);
            xv[u][0] = x[p[u]];
#pragma unroll
            for (int d = 0; d < 6; d++) xv[u][d + 1] = x[p[u] + nb[u].o[d]];
            bv[u] = b[p[u]];
        }
        __builtin_amdgcn_wave_barrier();  // the previous cells' entries have been read (one wave: LDS works in order)
#pragma unroll
        for (int u = 0; u < PU; u++)
#pragma unroll
            for (int m = 0; m < OPR_NST; m++) w[u * 64 * OPR_NST + lane + 64 * m] = av[u][m];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < PU; u++) {
            const double *A = w + (u * 64 + lane) * OPR_NST;
            const double a0 = A[sl.s[0]];
            double s = a0 * xv[u][0];
#pragma unroll
            for (int d = 0; d < 6; d++) {
                const double t = __builtin_fma(A[sl.s[d + 1]], xv[u][d + 1], s);
                s = (nb[u].has >> d) & 1 ? t : s;
            }
            if (!(fabs(a0) > 0.0)) s = xv[u][0];
            if (pw + u * stride + lane < g.N) {
                const double rv = bv[u] - s;
                r[p[u]] = rv;
                acc += rv * rv;
            }
        }
    }
    double t = block_sum(acc, sm);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// The exact operator as seven interior arrays (structure of arrays) for the
// nonsymmetric products of GMRES: o7[s * N + p], stencil slot s in the order
// centre, +x, -x, +y, -y, +z, -z. Identity rows (centre 0) get 1 and zero
// couplings; couplings out of a non-periodic box are 0. The same values the
// AoS products use, read coalesced.
__global__ void __launch_bounds__(NT) k_soa7(Geo g, Ghost gh, Slots sl, const double *__restrict__ opr,
                                             double *__restrict__ o7) {
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < g.N; p += (long long)gridDim.x * NT) {
        int i, j, k;
        decomp0(g, p, i, j, k);
        const double *A = opr + gidx(gh, i, j, k) * sl.nst;
        const double a0 = A[sl.s[0]];
        const bool pt = fabs(a0) > 0.0;
        o7[p] = pt ? a0 : 1.0;
        const bool in[6] = {nbp(i, g.n0, g.p0) >= 0, nbm(i, g.n0, g.p0) >= 0, nbp(j, g.n1, g.p1) >= 0,
                            nbm(j, g.n1, g.p1) >= 0, nbp(k, g.n2, g.p2) >= 0, nbm(k, g.n2, g.p2) >= 0};
        for (int q = 0; q < 6; q++) o7[(q + 1) * g.N + p] = (pt && in[q]) ? A[sl.s[q + 1]] : 0.0;
    }
}

// y = A x, or (b != nullptr) r = b - A x with partial ||r||^2 in part, from the
// seven-array form; the same sum order as k_exact_resid. 128^3: 42 us one cell
// at a time; 33 us now.
__global__ void __launch_bounds__(NT) k_apply7(Geo g, const double *__restrict__ o7, const double *__restrict__ b,
                                               const double *__restrict__ x, double *__restrict__ y,
                                               double *__restrict__ part) {
    __shared__ double sm[NT / 64];
    double acc = 0.0;
    const long long N = g.N, stride = (long long)gridDim.x * NT;
    for (long long p0 = blockIdx.x * (long long)NT + threadIdx.x; p0 < N; p0 += PU * stride) {
        int p[PU];
        Nb6 nb[PU];
        double ov[PU][7], xv[PU][7], bv[PU];
#pragma unroll
        for (int u = 0; u < PU; u++) {
            const long long q = p0 + u * stride;
            p[u] = q < N ? (int)q : (int)N - 1;
            int i, j, k;
            decomp0(g, p[u], i, j, k);
            nb[u] = nb6(g, i, j, k);
#pragma unroll
            for (int d = 0; d < 7; d++) ov[u][d] = o7[d * N + p[u]];
            xv[u][0] = x[p[u]];
#pragma unroll
            for (int d = 0; d < 6; d++) xv[u][d + 1] = x[p[u] + nb[u].o[d]];
            bv[u] = b ? b[p[u]] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < PU; u++) {
            double s = ov[u][0] * xv[u][0];
#pragma unroll
            for (int d = 0; d < 6; d++) {
                const double t = __builtin_fma(ov[u][d + 1], xv[u][d + 1], s);
                s = (nb[u].has >> d) & 1 ? t : s;
            }
            if (p0 + u * stride < N) {
                const double rv = b ? bv[u] - s : s;
                y[p[u]] = rv;
                if (b) acc += rv * rv;
            }
        }
    }
    if (part) {
        const double t = block_sum(acc, sm);
        if (threadIdx.x == 0) part[blockIdx.x] = t;
    }
}

// GMRES basis kernels. V holds nv vectors of n doubles, ld apart; at most
// GB_MAX vectors per launch (the caller splits longer bases). Partials of a
// launch (at most GPART blocks, the cap of grid_for) sit GPART apart.
constexpr int GB_MAX = 8;
constexpr int GPART = 1024;

// partial <w, V_i>, i < nv: parts[i * GPART + block]
__global__ void __launch_bounds__(NT) k_mdot(long long n, const double *__restrict__ w, const double *__restrict__ V,
                                             long long ld, int nv, double *__restrict__ parts) {
    __shared__ double sm[NT / 64];
    double acc[GB_MAX];
#pragma unroll
    for (int i = 0; i < GB_MAX; i++) acc[i] = 0.0;
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < n; p += (long long)gridDim.x * NT) {
        const double wv = w[p];
#pragma unroll
        for (int i = 0; i < GB_MAX; i++)
            if (i < nv) acc[i] += wv * V[i * ld + p];
    }
#pragma unroll
    for (int i = 0; i < GB_MAX; i++) {
        if (i >= nv) break;
        const double t = block_sum(acc[i], sm);
        if (threadIdx.x == 0) parts[i * GPART + blockIdx.x] = t;
    }
}

// out[i] = sum of parts[i * GPART + 0..nb-1] in block order, i < nv
__global__ void __launch_bounds__(NT) k_fin_multi(const double *__restrict__ parts, int nb, int nv,
                                                  double *__restrict__ out) {
    __shared__ double sm[NT / 64];
    for (int i = 0; i < nv; i++) {
        double v = 0.0;
        for (int b = threadIdx.x; b < nb; b += NT) v += parts[i * GPART + b];
        const double t = block_sum(v, sm);
        if (threadIdx.x == 0) out[i] = t;
    }
}

// w -= sum_i coef[i] V_i (i < nv); with sq, partial ||w||^2 of the result
__global__ void __launch_bounds__(NT) k_gs_update(long long n, double *__restrict__ w, const double *__restrict__ V,
                                                  long long ld, int nv, const double *__restrict__ coef,
                                                  double *__restrict__ sq) {
    __shared__ double sm[NT / 64];
    double c[GB_MAX];
#pragma unroll
    for (int i = 0; i < GB_MAX; i++) c[i] = i < nv ? coef[i] : 0.0;
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < n; p += (long long)gridDim.x * NT) {
        double v = w[p];
#pragma unroll
        for (int i = 0; i < GB_MAX; i++)
            if (i < nv) v -= c[i] * V[i * ld + p];
        w[p] = v;
        acc += v * v;
    }
    if (sq) {
        const double t = block_sum(acc, sm);
        if (threadIdx.x == 0) sq[blockIdx.x] = t;
    }
}

// x += sum_i coef[i] Z_i (i < nv)
__global__ void __launch_bounds__(NT) k_lincomb(long long n, double *__restrict__ x, const double *__restrict__ Z,
                                                long long ld, int nv, const double *__restrict__ coef) {
    double c[GB_MAX];
#pragma unroll
    for (int i = 0; i < GB_MAX; i++) c[i] = i < nv ? coef[i] : 0.0;
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < n; p += (long long)gridDim.x * NT) {
        double v = x[p];
#pragma unroll
        for (int i = 0; i < GB_MAX; i++)
            if (i < nv) v += c[i] * Z[i * ld + p];
        x[p] = v;
    }
}

__global__ void __launch_bounds__(NT) k_scale_to(long long n, const double *__restrict__ s, double f,
                                                 double *__restrict__ d) {
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < n; p += (long long)gridDim.x * NT) d[p] = s[p] * f;
}

__global__ void __launch_bounds__(NT) k_sumsq(long long n, const double *__restrict__ x, double *__restrict__ part) {
    __shared__ double sm[NT / 64];
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < n; p += (long long)gridDim.x * NT) acc += x[p] * x[p];
    double t = block_sum(acc, sm);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

template <typename Tx, typename Ty>
__global__ void __launch_bounds__(NT) k_dot(long long n, const Tx *__restrict__ x, const Ty *__restrict__ y,
                                            double *__restrict__ part) {
    __shared__ double sm[NT / 64];
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)NT + threadIdx.x; p < n; p += (long long)gridDim.x * NT)
        acc += (double)x[p] * (double)y[p];
    double t = block_sum(acc, sm);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// The PCG vector kernels walk the vectors in pairs: one 16-byte load per FP64
// array (8 bytes for an FP32 one) per thread and step. An odd last element is
// taken by thread 0 of block 0.
struct alignas(16) D2 {
    double a, b;
};
struct alignas(8) F2 {
    float a, b;
};

template <typename Tz>
struct Pair;
template <>
struct Pair<double> {
    typedef D2 type;
};
template <>
struct Pair<float> {
    typedef F2 type;
};

// x += alpha p ; r -= alpha q ; partial ||r||^2 ; optional FP32 copy of r.
// Tp: the type p is stored in (FP32 in the mixed solve)
template <typename Tp>
__global__ void __launch_bounds__(NT) k_update_xr(long long n, double *__restrict__ x, double *__restrict__ r,
                                                  const Tp *__restrict__ p, const double *__restrict__ q,
                                                  const double *__restrict__ scal, float *__restrict__ r32,
                                                  double *__restrict__ part) {
    typedef typename Pair<Tp>::type PP;
    __shared__ double sm[NT / 64];
    const double a = scal[S_ALPHA];
    double acc = 0.0;
    const long long n2 = n >> 1;
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n2; i += (long long)gridDim.x * NT) {
        D2 rv = reinterpret_cast<const D2 *>(r)[i];
        if (a != 0.0) {
            D2 xv = reinterpret_cast<const D2 *>(x)[i];
            const PP pv = reinterpret_cast<const PP *>(p)[i];
            const D2 qv = reinterpret_cast<const D2 *>(q)[i];
            xv.a += a * (double)pv.a;
            xv.b += a * (double)pv.b;
            rv.a -= a * qv.a;
            rv.b -= a * qv.b;
            reinterpret_cast<D2 *>(x)[i] = xv;
            reinterpret_cast<D2 *>(r)[i] = rv;
        }
        acc += rv.a * rv.a;
        acc += rv.b * rv.b;
        if (r32) reinterpret_cast<F2 *>(r32)[i] = F2{(float)rv.a, (float)rv.b};
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const long long i = n - 1;
        double rv = r[i];
        if (a != 0.0) {
            x[i] += a * (double)p[i];
            rv -= a * q[i];
            r[i] = rv;
        }
        acc += rv * rv;
        if (r32) r32[i] = (float)rv;
    }
    double t = block_sum(acc, sm);
    if (threadIdx.x == 0) part[blockIdx.x] = t;
}

// <r,z> and (optionally) <z,q>
template <typename Tz>
__global__ void __launch_bounds__(NT) k_dot_rz(long long n, const double *__restrict__ r, const Tz *__restrict__ z,
                                               const double *__restrict__ q, double *__restrict__ p_rz,
                                               double *__restrict__ p_zq) {
    typedef typename Pair<Tz>::type P;
    __shared__ double sm[NT / 64];
    double a = 0.0, b = 0.0;
    const long long n2 = n >> 1;
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n2; i += (long long)gridDim.x * NT) {
        const P zv = reinterpret_cast<const P *>(z)[i];
        const D2 rv = reinterpret_cast<const D2 *>(r)[i];
        const double z0 = (double)zv.a, z1 = (double)zv.b;
        a += rv.a * z0;
        a += rv.b * z1;
        if (q) {
            const D2 qv = reinterpret_cast<const D2 *>(q)[i];
            b += z0 * qv.a;
            b += z1 * qv.b;
        }
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const long long i = n - 1;
        const double zv = (double)z[i];
        a += r[i] * zv;
        if (q) b += zv * q[i];
    }
    double t = block_sum(a, sm);
    if (threadIdx.x == 0) p_rz[blockIdx.x] = t;
    if (q) {
        double u = block_sum(b, sm);
        if (threadIdx.x == 0) p_zq[blockIdx.x] = u;
    }
}

// p = z + beta p (copy: p = z), formed in FP64 and stored as Tp: FP32 in the
// mixed solve, whose directions come from the FP32 cycle (the x and r updates
// use the stored p exactly, so they stay consistent with each other)
template <typename Tz, typename Tp>
__global__ void __launch_bounds__(NT) k_update_p(long long n, Tp *__restrict__ p, const Tz *__restrict__ z,
                                                 const double *__restrict__ scal, int copy) {
    typedef typename Pair<Tz>::type P;
    typedef typename Pair<Tp>::type PP;
    const double be = copy ? 0.0 : scal[S_BETA];
    const long long n2 = n >> 1;
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n2; i += (long long)gridDim.x * NT) {
        const P zv = reinterpret_cast<const P *>(z)[i];
        double a, b;
        if (copy) {
            a = (double)zv.a;
            b = (double)zv.b;
        } else {
            const PP pv = reinterpret_cast<const PP *>(p)[i];
            a = (double)zv.a + be * (double)pv.a;
            b = (double)zv.b + be * (double)pv.b;
        }
        reinterpret_cast<PP *>(p)[i] = PP{(Tp)a, (Tp)b};
    }
    if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
        const long long i = n - 1;
        const double zv = (double)z[i];
        p[i] = (Tp)(copy ? zv : zv + be * (double)p[i]);
    }
}

__global__ void __launch_bounds__(NT) k_copy(long long n, const double *__restrict__ s, double *__restrict__ d) {
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n; i += (long long)gridDim.x * NT) d[i] = s[i];
}

__global__ void __launch_bounds__(NT) k_zero64(long long n, double *__restrict__ d) {
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n; i += (long long)gridDim.x * NT) d[i] = 0.0;
}

// t = r - t
__global__ void __launch_bounds__(NT) k_sub_from(long long n, const double *__restrict__ r, double *__restrict__ t) {
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n; i += (long long)gridDim.x * NT) t[i] = r[i] - t[i];
}

// z += e
__global__ void __launch_bounds__(NT) k_add(long long n, double *__restrict__ z, const double *__restrict__ e) {
    for (long long i = blockIdx.x * (long long)NT + threadIdx.x; i < n; i += (long long)gridDim.x * NT) z[i] += e[i];
}

__device__ __forceinline__ double sum_parts(const double *__restrict__ parts, int n, double *sm) {
    double s = 0.0;
    for (int q = threadIdx.x; q < n; q += NT) s += parts[q];
    return block_sum(s, sm);
}

__device__ __forceinline__ double max_parts(const double *__restrict__ parts, int n, double *sm) {
    double s = 0.0;
    for (int q = threadIdx.x; q < n; q += NT) s = fmax(s, parts[q]);
    return block_max(s, sm);
}

__global__ void __launch_bounds__(NT) k_fin_sum(const double *__restrict__ parts, int n, double *__restrict__ scal,
                                                int slot) {
    __shared__ double sm[NT / 64];
    double s = sum_parts(parts, n, sm);
    if (threadIdx.x == 0) scal[slot] = s;
}

// scal[slot + v] = sum of parts[v * MAX_PARTS + 0..n-1], v < nv, each in k_fin_sum's order
__global__ void __launch_bounds__(NT) k_fin_sums(const double *__restrict__ parts, int n, int nv,
                                                 double *__restrict__ scal, int slot) {
    __shared__ double sm[NT / 64];
    for (int v = 0; v < nv; v++) {
        double s = sum_parts(parts + (size_t)v * MAX_PARTS, n, sm);
        if (threadIdx.x == 0) scal[slot + v] = s;
    }
}

__global__ void __launch_bounds__(NT) k_fin_max(const double *__restrict__ parts, int n, double *__restrict__ scal,
                                                int slot) {
    __shared__ double sm[NT / 64];
    double s = max_parts(parts, n, sm);
    if (threadIdx.x == 0) scal[slot] = s;
}

// alpha = rho / <p,Ap>; 0 and a flag on breakdown. The SpMV leaves up to
// MAX_PARTS partials, so this finalize runs 1024 threads (8 loads each at
// 256^3 instead of 32), in a fixed order.
constexpr int NT_FIN = 1024;
__global__ void __launch_bounds__(NT_FIN) k_fin_alpha(const double *__restrict__ parts, int n,
                                                      double *__restrict__ scal, int *__restrict__ flags) {
    __shared__ double sm[NT_FIN / 64];
    double v = 0.0;
    for (int q = threadIdx.x; q < n; q += NT_FIN) v += parts[q];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double pq = 0.0;
        for (int w = 0; w < NT_FIN / 64; w++) pq += sm[w];
        double rho = scal[S_RHO];
        double a = rho / pq;
        if (!(pq > 0.0) || !(rho > 0.0) || !isfinite(a)) {
            a = 0.0;
            flags[0] |= 1;
        }
        scal[S_PQ] = pq;
        scal[S_ALPHA] = a;
    }
}

// rho = <r,z> after a restart
__global__ void __launch_bounds__(NT) k_fin_rho(const double *__restrict__ parts, int n, double *__restrict__ scal,
                                                int *__restrict__ flags, int first) {
    __shared__ double sm[NT / 64];
    double rz = sum_parts(parts, n, sm);
    if (threadIdx.x == 0) {
        if (!(rz > 0.0) || !isfinite(rz)) flags[0] |= 2;
        scal[S_RHO] = rz;
        if (first) scal[S_RHO0] = rz;
    }
}

// beta (plain: <r+,z+>/<r,z>; flexible: -alpha <z+,q>/<r,z>)
__global__ void __launch_bounds__(NT) k_fin_beta(const double *__restrict__ p_rz, const double *__restrict__ p_zq,
                                                 int n, double *__restrict__ scal, int *__restrict__ flags,
                                                 int flexible) {
    __shared__ double sm[NT / 64];
    double rz = sum_parts(p_rz, n, sm);
    double zq = flexible ? sum_parts(p_zq, n, sm) : 0.0;
    if (threadIdx.x == 0) {
        double rho = scal[S_RHO];
        double be = flexible ? -scal[S_ALPHA] * zq / rho : rz / rho;
        if (!(rz > 0.0) || !isfinite(be)) {
            be = 0.0;
            flags[0] |= 2;
        }
        scal[S_BETA] = be;
        scal[S_RHO] = rz;
    }
}

__global__ void k_clear_flags(int *flags) {
    if (threadIdx.x == 0) flags[0] = 0;
}

// workgroups of a streaming kernel without partial sums, `per` cells a thread
int stream_blocks(long long n, int per) {
    const long long b = (n + (long long)NT * per - 1) / ((long long)NT * per);
    return (int)(b < 1 ? 1 : (b > 65536 ? 65536 : b));
}

double now_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

}  // namespace

// ====================================================================== handle

// Host staging of the host entry points (ngap_solve). The caller's arrays are
// pageable. They move through pinned chunks: STG_THREADS host threads each own
// a contiguous part of the array, two pinned chunks and a HIP stream, and copy
// chunk by chunk between pageable and pinned memory while the DMA engine moves
// the other chunk of the pair.
constexpr int STG_THREADS = 4;
constexpr size_t STG_CHUNK = (size_t)4 << 20;  // bytes per pinned chunk
struct Staging {
    char *pin = nullptr;  // 2 * STG_THREADS chunks
    hipStream_t st[STG_THREADS] = {};
    hipEvent_t ev[STG_THREADS][2] = {};
    bool ready = false;
};

struct ngap_t {
    ngap_grid g{};
    int nst = 0;
    std::vector<int> stc;
    int method = 0;
    Slots slots{};
    bool init_done = false, setup_done = false;
    int maxit = 100;
    double rcvg = 1e-10;
    int maxlevel = 0;
    ngap_opts opts{};
    int device = 0;
    hipStream_t stream = nullptr;
    Ghost gh{};
    long long nghost = 0;
    Geo g0{};
    std::vector<Level> lev;
    int nlev = 0;
    double *opr = nullptr;  // own ghosted copy of the exact operator
    unsigned char *part = nullptr;
    double *rhs_g = nullptr, *sol_g = nullptr;  // ghosted staging for host variants
    double *b = nullptr, *x = nullptr, *r = nullptr, *z = nullptr, *p = nullptr, *q = nullptr;
    float *r32 = nullptr, *z32 = nullptr;
    double *parts = nullptr;  // 4 * MAX_PARTS
    double *scal = nullptr;
    int *flags = nullptr;
    double *h_scal = nullptr;  // pinned
    int *h_flags = nullptr;    // pinned, inside the h_scal allocation
    hipEvent_t ev_scal = nullptr;  // marks the copy of the scalars into h_scal
    double *Ainv = nullptr;
    int nc = 0;
    int coarse_dense = 0, coarse_singular = 0;
    int apply_parts = 0;  // partial sums written by the fine-level SpMV
    hipGraphExec_t vc_graph[2] = {nullptr, nullptr};  // V-cycle per precision (0 FP64, 1 FP32)
    std::vector<long long> vc_key[2];                  // what each graph recorded (cycle_key)
    ngap_stats st{};
    long long dev_bytes = 0;
    std::vector<void *> base_allocs;
    // correction stage (ngap_set_stage)
    ngap_stage_fn stage_fn = nullptr;
    void *stage_ctx = nullptr;
    int stage_flags = 0, stage_iters = 0;
    double *st_t = nullptr, *st_e = nullptr;  // stage input and output, allocated on first use
    // flexible GMRES (method NGAP_GMRES_PFMG): Krylov basis V (kdim+1 vectors),
    // preconditioned directions Z (kdim), and the per-step scalars
    int kdim = 0;
    double *gV = nullptr, *gZ = nullptr;
    double *o7 = nullptr;    // the exact operator as seven interior arrays
    double *gm = nullptr;    // device scalars: [0,64) dots, [64,128) second-pass dots, 128 ||w||^2, [192,256) y
    double *h_gm = nullptr;  // pinned copy
    int fail_alloc = 0;      // > 0: the fail_alloc-th next device allocation fails (ngapt_fail_alloc)
    Staging stg;             // pinned staging of ngap_solve, made on its first call
    int relax_keep = 1;      // levels 0..relax_keep-1 are always smoothed (set_relax)
    bool x_zero = false;     // the guess of the solve in work is zero (counted with check_finite)
    bool p32 = false;        // p holds FP32 values (the mixed solve's directions), set at each restart
    long long zero_chunks = 0;  // guess chunks of the last ngap_solve found all zero (not copied)
    // the last setup completed with these options; its levels and coarsening
    // directions are then the first guess of the next setup's hierarchy
    bool spec_valid = false;
    int spec_maxlevel = 0, spec_coarsest = 0;
};

namespace {

hipError_t g_last_hip = hipSuccess;

#define HIPCHK(expr)                                       \
    do {                                                   \
        hipError_t e_ = (expr);                            \
        if (e_ != hipSuccess) {                            \
            g_last_hip = e_;                               \
            return e_ == hipErrorOutOfMemory ? NGAP_ERR_ALLOC : NGAP_ERR_HIP; \
        }                                                  \
    } while (0)

int dmalloc(ngap_t *h, void **ptr, size_t bytes) {
    *ptr = nullptr;
    if (bytes == 0) bytes = 8;
    if (h->fail_alloc > 0 && --h->fail_alloc == 0) return NGAP_ERR_ALLOC;  // injected by a test
    hipError_t e = hipMalloc(ptr, bytes);
    if (e != hipSuccess) {
        g_last_hip = e;
        *ptr = nullptr;
        return NGAP_ERR_ALLOC;
    }
    h->dev_bytes += (long long)bytes;
    return 0;
}

void dfree(ngap_t *h, void *ptr, size_t bytes) {
    if (ptr) {
        (void)hipFree(ptr);
        h->dev_bytes -= (long long)bytes;
    }
}

// coefficients and the second iterate buffer on every level; transfer
// weights, right-hand side and final iterate on coarse levels only
template <typename T>
int alloc_lvl_data(ngap_t *h, LevelData<T> &D, long long N, bool coarse) {
    size_t b = sizeof(T) * (size_t)N;
    int rc = 0;
    rc |= dmalloc(h, (void **)&D.c, b);
    rc |= dmalloc(h, (void **)&D.a0, b);
    rc |= dmalloc(h, (void **)&D.a1, b);
    rc |= dmalloc(h, (void **)&D.a2, b);
    rc |= dmalloc(h, (void **)&D.w, b);
    if (coarse) {
        rc |= dmalloc(h, (void **)&D.pm, b);
        rc |= dmalloc(h, (void **)&D.pp, b);
        rc |= dmalloc(h, (void **)&D.f, b);
        rc |= dmalloc(h, (void **)&D.v, b);
    }
    return rc ? NGAP_ERR_ALLOC : 0;
}

template <typename T>
void free_lvl_data(ngap_t *h, LevelData<T> &D, long long N) {
    size_t b = sizeof(T) * (size_t)N;
    for (T *q : {D.c, D.a0, D.a1, D.a2, D.w, D.pm, D.pp, D.f, D.v}) dfree(h, q, b);
    D = LevelData<T>();
}

void free_level(ngap_t *h, Level &L) {
    free_lvl_data(h, L.d, L.g.N);
    free_lvl_data(h, L.s, L.g.N);
}

void destroy_graphs(ngap_t *h);

void free_all(ngap_t *h) {
    destroy_graphs(h);
    for (auto &L : h->lev) free_level(h, L);
    h->lev.clear();
    h->nlev = 0;
    if (h->Ainv) {
        dfree(h, h->Ainv, sizeof(double) * (size_t)h->nc * h->nc);
        h->Ainv = nullptr;
    }
    size_t N = (size_t)h->g0.N;
    dfree(h, h->opr, sizeof(double) * (size_t)h->nghost * h->nst);
    dfree(h, h->part, N);
    dfree(h, h->rhs_g, sizeof(double) * (size_t)h->nghost);
    dfree(h, h->sol_g, sizeof(double) * (size_t)h->nghost);
    for (double **v : {&h->b, &h->x, &h->r, &h->z, &h->p, &h->q}) {
        dfree(h, *v, sizeof(double) * N);
        *v = nullptr;
    }
    dfree(h, h->r32, sizeof(float) * N);
    dfree(h, h->z32, sizeof(float) * N);
    dfree(h, h->st_t, sizeof(double) * N);
    dfree(h, h->st_e, sizeof(double) * N);
    h->st_t = h->st_e = nullptr;
    dfree(h, h->gV, sizeof(double) * N * (h->kdim + 1));
    dfree(h, h->gZ, sizeof(double) * N * h->kdim);
    dfree(h, h->gm, sizeof(double) * 256);
    dfree(h, h->o7, sizeof(double) * N * 7);
    h->gV = h->gZ = h->gm = h->o7 = nullptr;
    h->kdim = 0;
    dfree(h, h->parts, sizeof(double) * 4 * MAX_PARTS);
    dfree(h, h->scal, SCAL_BYTES);  // flags share the allocation
    h->opr = nullptr;
    h->part = nullptr;
    h->rhs_g = h->sol_g = nullptr;
    h->r32 = h->z32 = nullptr;
    h->parts = h->scal = nullptr;
    h->flags = nullptr;
}

// fine-level and PCG buffers (depend only on the grid)
int ensure_base(ngap_t *h) {
    if (h->opr) return 0;
    size_t N = (size_t)h->g0.N;
    int rc = 0;
    rc |= dmalloc(h, (void **)&h->opr, sizeof(double) * (size_t)h->nghost * h->nst);
    rc |= dmalloc(h, (void **)&h->part, N);
    rc |= dmalloc(h, (void **)&h->rhs_g, sizeof(double) * (size_t)h->nghost);
    rc |= dmalloc(h, (void **)&h->sol_g, sizeof(double) * (size_t)h->nghost);
    for (double **v : {&h->b, &h->x, &h->r, &h->z, &h->p, &h->q}) rc |= dmalloc(h, (void **)v, sizeof(double) * N);
    rc |= dmalloc(h, (void **)&h->r32, sizeof(float) * N);
    rc |= dmalloc(h, (void **)&h->z32, sizeof(float) * N);
    rc |= dmalloc(h, (void **)&h->parts, sizeof(double) * 4 * MAX_PARTS);
    rc |= dmalloc(h, (void **)&h->scal, SCAL_BYTES);
    if (h->scal) h->flags = reinterpret_cast<int *>(h->scal + NSCAL_ALLOC);
    if (rc) {
        free_all(h);
        return NGAP_ERR_ALLOC;
    }
    if (!h->h_scal) {
        HIPCHK(hipHostMalloc((void **)&h->h_scal, SCAL_BYTES, hipHostMallocDefault));
        h->h_flags = reinterpret_cast<int *>(h->h_scal + NSCAL_ALLOC);
    }
    HIPCHK(hipMemsetAsync(h->scal, 0, SCAL_BYTES, h->stream));
    return 0;
}

int read_scal(ngap_t *h) {
    // the scalars and the flags behind them, one copy
    HIPCHK(hipMemcpyAsync(h->h_scal, h->scal, SCAL_BYTES, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    return 0;
}

// Which levels the V-cycle smooths (skipped relaxation, after PFMG's SkipRelax,
// with this project's rule): with skip set, a level l with 0 < l < nlev-1 is
// smoothed only when its couplings are isotropic: over the directions with
// n_d > 1 and s_d = sum |a_d| > 0 (the strengths of the coarsening choice),
// max s_d <= 2 min s_d (with a 1e-6 relative margin, so a ratio of 2 up to the
// rounding of the sums counts as isotropic in any summation order), or fewer
// than two such directions. Semicoarsening an
// isotropic grid in x, y, z takes the strengths (1,1,1) -> (1/2,2,2) ->
// (1,1,4) -> (2,2,2), so every third level is smoothed, as in full
// coarsening. A skipped level restricts its right-hand side unchanged on the
// way down (v = 0) and takes v = P v_coarse on the way up. The finest level is
// always smoothed, the coarsest always solved, and levels below relax_keep
// smoothed (all of them on a locally anisotropic operator).
// Skipping the intermediate levels suits isotropic operators. A locally
// anisotropic fine operator (more than 10% of its cells anisotropic by
// k_aniso_count's measure: a stretched wall grid) smooths every level:
// skipping took the channel from 13 to 26 iterations, and keeping the first
// coarsening round smoothed still to 17 at 256^3. The interface cells of a
// two-phase operator are few, and its gate stays open.
int skip_gate(double cells, double aniso) { return cells > 0.0 && aniso * 10.0 <= cells; }

void set_relax(ngap_t *h, int skip) {
    for (int l = 0; l < h->nlev; l++) {
        Level &L = h->lev[l];
        L.relax = true;
        if (!skip || l < h->relax_keep || l == h->nlev - 1) continue;
        const int n[3] = {L.g.n0, L.g.n1, L.g.n2};
        double smin = INFINITY, smax = 0.0;
        int cnt = 0;
        for (int d = 0; d < 3; d++) {
            if (n[d] < 2 || !(L.str[d] > 0.0)) continue;
            cnt++;
            smin = std::min(smin, L.str[d]);
            smax = std::max(smax, L.str[d]);
        }
        L.relax = cnt < 2 || smax <= 2.0 * (1.0 + 1e-6) * smin;
    }
}

int can_coarsen(const Geo &g, int d) {
    int n = d == 0 ? g.n0 : (d == 1 ? g.n1 : g.n2);
    int per = d == 0 ? g.p0 : (d == 1 ? g.p1 : g.p2);
    if (per) return (n % 4) == 0;  // coarse periodic length stays even (red/black colouring)
    return n >= 2;
}

// Coarsening direction of a level from its strengths sv[d] = sum |a_d|: the
// strongest direction that can be coarsened (ties within a 1e-6 relative
// margin to the lowest d), -1 when none can.
int pick_dir(const Geo &g, const double *sv) {
    double str[3];
    for (int d = 0; d < 3; d++) str[d] = can_coarsen(g, d) ? sv[d] : -1.0;
    int best = -1;
    for (int d = 0; d < 3; d++) {
        if (str[d] < 0) continue;
        if (best < 0 || str[d] > str[best] * (1.0 + 1e-6)) best = d;
    }
    return best;
}

// ---------------------------------------------------------------- coarsest (host)

// sum of a[k] b[k] over k in [lo, hi), in four interleaved partial sums
// (the compiler keeps a single running sum in order and cannot vectorise it)
double dot4(const double *a, const double *b, int lo, int hi) {
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int k = lo;
    for (; k + 4 <= hi; k += 4) {
        s0 += a[k] * b[k];
        s1 += a[k + 1] * b[k + 1];
        s2 += a[k + 2] * b[k + 2];
        s3 += a[k + 3] * b[k + 3];
    }
    for (; k < hi; k++) s0 += a[k] * b[k];
    return (s0 + s1) + (s2 + s3);
}

// the coarsest inverse's buffer for n cells
int ensure_ainv(ngap_t *h, int n) {
    if (h->Ainv && h->nc != n) {
        dfree(h, h->Ainv, sizeof(double) * (size_t)h->nc * h->nc);
        h->Ainv = nullptr;
    }
    h->nc = n;
    if (!h->Ainv && dmalloc(h, (void **)&h->Ainv, sizeof(double) * (size_t)n * n)) return NGAP_ERR_ALLOC;
    return 0;
}

// Dense coarsest operator -> (pseudo-)inverse, FP64, on the host (coarsest
// levels of more than COARSE_LDS_MAX cells; k_coarse_inverse below that).
int build_coarsest_inverse(ngap_t *h) {
    int rc;
    Level &C = h->lev[h->nlev - 1];
    const Geo &g = C.g;
    int n = (int)g.N;
    std::vector<double> c(n), a0(n), a1(n), a2(n);
    HIPCHK(hipMemcpyAsync(c.data(), C.d.c, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipMemcpyAsync(a0.data(), C.d.a0, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipMemcpyAsync(a1.data(), C.d.a1, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipMemcpyAsync(a2.data(), C.d.a2, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    const double *a[3] = {a0.data(), a1.data(), a2.data()};
    const int n3[3] = {g.n0, g.n1, g.n2}, p3[3] = {g.p0, g.p1, g.p2};
    std::vector<double> M((size_t)n * n, 0.0);
    double ssum = 0.0, csum = 0.0;
    auto lin = [&](int i, int j, int k) { return (long long)i + (long long)g.n0 * ((long long)j + (long long)g.n1 * k); };
    for (int k = 0; k < g.n2; k++)
        for (int j = 0; j < g.n1; j++)
            for (int i = 0; i < g.n0; i++) {
                long long p = lin(i, j, k);
                M[p * n + p] += c[p];
                int c3[3] = {i, j, k};
                double rs = c[p];
                for (int d = 0; d < 3; d++) {
                    int qm = c3[d] > 0 ? c3[d] - 1 : (p3[d] ? n3[d] - 1 : -1);
                    if (qm >= 0) {
                        int e3[3] = {i, j, k};
                        e3[d] = qm;
                        long long pq = lin(e3[0], e3[1], e3[2]);
                        M[p * n + pq] += a[d][p];
                        M[pq * n + p] += a[d][p];
                    }
                    rs += a[d][p];
                    int qp = c3[d] < n3[d] - 1 ? c3[d] + 1 : (p3[d] ? 0 : -1);
                    if (qp >= 0) {
                        int e3[3] = {i, j, k};
                        e3[d] = qp;
                        rs += a[d][lin(e3[0], e3[1], e3[2])];
                    }
                }
                ssum += std::fabs(rs);
                csum += std::fabs(c[p]);
            }
    h->coarse_singular = ssum <= 1e-10 * csum;
    if (h->coarse_singular) {
        double gam = csum / ((double)n * n);
        for (auto &m : M) m += gam;
    }
    // Cholesky (lower), then A^-1 = W^T W with W = L^-1. Rows are contiguous,
    // so every inner product runs over contiguous memory (dot4).
    std::vector<double> L((size_t)n * n, 0.0);
    for (int j = 0; j < n; j++) {
        const double *Lj = &L[(size_t)j * n];
        double s = M[(size_t)j * n + j] - dot4(Lj, Lj, 0, j);
        if (!(s > 0.0)) return NGAP_ERR_COARSE;
        double ljj = std::sqrt(s);
        L[(size_t)j * n + j] = ljj;
        for (int i = j + 1; i < n; i++)
            L[(size_t)i * n + j] = (M[(size_t)i * n + j] - dot4(&L[(size_t)i * n], Lj, 0, j)) / ljj;
    }
    // Y[col][i] = W[i][col] (zero for i < col): forward substitution on e_col
    std::vector<double> Y((size_t)n * n, 0.0), X((size_t)n * n, 0.0);
    for (int col = 0; col < n; col++) {
        double *y = &Y[(size_t)col * n];
        for (int i = col; i < n; i++) {
            const double *Li = &L[(size_t)i * n];
            y[i] = ((i == col ? 1.0 : 0.0) - dot4(Li, y, col, i)) / Li[i];
        }
    }
    for (int a = 0; a < n; a++)
        for (int b = a; b < n; b++) {
            const double v = dot4(&Y[(size_t)a * n], &Y[(size_t)b * n], b, n);
            X[(size_t)a * n + b] = v;
            X[(size_t)b * n + a] = v;
        }
    if ((rc = ensure_ainv(h, n))) return rc;
    HIPCHK(hipMemcpy(h->Ainv, X.data(), sizeof(double) * (size_t)n * n, hipMemcpyHostToDevice));
    return 0;
}

// ---------------------------------------------------------------- V-cycle

template <typename T>
LevelData<T> &data(Level &L);
template <>
LevelData<double> &data<double>(Level &L) { return L.d; }
template <>
LevelData<float> &data<float>(Level &L) { return L.s; }

// Coarsest level: dense (pseudo-)inverse, or 8 RB/BR sweep pairs from zero.
// The result lands in v.
template <typename T>
void coarse_solve(ngap_t *h, const T *f, T *v) {
    Level &C = h->lev[h->nlev - 1];
    LevelData<T> &D = data<T>(C);
    if (h->coarse_dense) {
        launch_dense<T, T>(h->stream, (int)C.g.N, h->Ainv, f, v);
    } else {
        launch_sweep<T>(h->stream, C.g, D.c, D.a0, D.a1, D.a2, f, nullptr, D.w, 0);
        launch_sweep<T>(h->stream, C.g, D.c, D.a0, D.a1, D.a2, f, D.w, v, 1);
        for (int s = 1; s < 8; s++) {
            launch_sweep<T>(h->stream, C.g, D.c, D.a0, D.a1, D.a2, f, v, D.w, 0);
            launch_sweep<T>(h->stream, C.g, D.c, D.a0, D.a1, D.a2, f, D.w, v, 1);
        }
    }
}

// First level of the small-level bottom (k_bottom) in precision T, or nlev when
// the bottom is not used: it needs the dense coarsest solve, at least one
// smoothing level below the fine level, at most BOT_MAX_LEVELS levels, and
// levels that fit it.
template <typename T>
int bottom_start(const ngap_t *h) {
    const int nl = h->nlev;
    if (!h->coarse_dense || nl < 3) return nl;
    std::vector<Geo> g;
    for (const Level &L : h->lev) g.push_back(L.g);
    int lb = nl - 1;
    while (lb - 1 >= 1 && nl - (lb - 1) <= BOT_MAX_LEVELS && bottom_fits<T>(&g[lb - 1], nl - (lb - 1))) lb--;
    return lb <= nl - 2 ? lb : nl;
}

template <typename T>
void launch_bottom_levels(ngap_t *h, int lb) {
    BotArgs<T> a{};
    a.nlev = h->nlev - lb;
    a.npre = h->opts.nu_pre;
    a.npost = h->opts.nu_post;
    a.Ainv = h->Ainv;
    for (int q = 0; q < a.nlev; q++) {
        Level &L = h->lev[lb + q];
        LevelData<T> &D = data<T>(L);
        a.L[q] = BotLevel<T>{L.g, BotDir{L.cdir}, L.relax ? 1 : 0, D.c, D.a0, D.a1, D.a2, D.pm, D.pp, D.f, D.v, 0.0f, 0.0f};
    }
    launch_bottom<T>(h->stream, a);
}

// Levels whose first pre-smoothing sweep (from a zero iterate) runs as the
// whole-row sweep kernel rather than the stencil form: rows of <= 128 cells,
// >= 2^20 cells. The stencil reads f and c at every neighbour to form f / c;
// the sweep forms it once per cell and passes it through LDS (256^3 channel,
// mixed: 27.40 against 27.20 ms per solve). Both give the same bits.
constexpr long long ZSWEEP_MIN_CELLS = 1LL << 20;

// The three transfers below level l as one launch: l + 1 and l + 2 are skipped
// levels, l + 3 is at most `top`, and the three directions differ (order 0: not so).
template <typename T>
struct Skip3 {
    Geo g[4];
    const T *pm[3], *pp[3];
    int order = 0;
    Skip3(ngap_t *h, int l, int top) {
        if (l + 3 > top || h->lev[l + 1].relax || h->lev[l + 2].relax) return;
        int dirs[3];
        g[0] = h->lev[l].g;
        for (int i = 0; i < 3; i++) {
            dirs[i] = h->lev[l + i].cdir;
            g[i + 1] = h->lev[l + i + 1].g;
            LevelData<T> &D = data<T>(h->lev[l + i + 1]);
            pm[i] = D.pm;
            pp[i] = D.pp;
        }
        order = chain_order(dirs);
    }
};

// One V(nu_pre, nu_post) cycle from a zero guess: v0 = M f0.
// Sweeps are out of place; on each level the iterate alternates between the
// level's two buffers so that the last post-smoothing sweep lands in the
// final buffer (v0 on the fine level, D.v on coarse levels). The levels from
// bottom_start() down run inside one workgroup (k_bottom), result in D.v.
template <typename T>
void vcycle(ngap_t *h, const T *f0, T *v0) {
    const int nl = h->nlev;
    hipStream_t s = h->stream;
    const int npre = h->opts.nu_pre, npost = h->opts.nu_post;
    // On the levels of pairs_on the post-smoothing sweeps run in fused pairs
    // (one launch each) plus a single one for an odd count; every launch
    // switches the level's buffer.
    auto post_launches = [&](const Level &L) { return pairs_on<T>(L.g) ? npost / 2 + (npost & 1) : npost; };
    // pre-smoothing on those levels: the first two sweeps (from a zero
    // iterate) as one pair launch, the rest as in the post-smoothing
    auto pre_launches = [&](const Level &L) {
        if (!pairs_on<T>(L.g) || npre < 2) return npre;
        return 1 + (npre - 2) / 2 + ((npre - 2) & 1);
    };
    const int lb = bottom_start<T>(h);
    const int top = lb < nl ? lb : nl - 1;  // first level below the per-level loop
    std::vector<T *> pre(nl);
    std::vector<char> bridged(nl, 0);  // skipped levels that a Skip3 launch passes over
    auto restrict_from = [&](int l, const T *r) {
        const Skip3<T> k(h, l, top);
        if (k.order) {
            launch_gather3<T>(s, k.g, k.order, k.pm, k.pp, r, data<T>(h->lev[l + 3]).f);
            bridged[l + 1] = bridged[l + 2] = 1;
            return;
        }
        LevelData<T> &DC = data<T>(h->lev[l + 1]);
        launch_gather<T>(s, h->lev[l].g, h->lev[l + 1].g, h->lev[l].cdir, r, DC.pm, DC.pp, DC.f);
    };
    auto prolong_to = [&](int l, const T *vin, T *vout) {
        if (l + 1 < nl && bridged[l + 1]) {
            const Skip3<T> k(h, l, top);
            launch_prolong3<T>(s, k.g, k.order, k.pm, k.pp, data<T>(h->lev[l + 3]).v, vin, vout);
            return;
        }
        LevelData<T> &DC = data<T>(h->lev[l + 1]);
        launch_prolong_to<T>(s, h->lev[l].g, h->lev[l + 1].g, h->lev[l].cdir, DC.pm, DC.pp, DC.v, vin, vout);
    };
    for (int l = 0; l < top; l++) {
        if (bridged[l]) continue;
        Level &L = h->lev[l];
        LevelData<T> &D = data<T>(L);
        const T *f = l == 0 ? f0 : D.f;
        T *fin = l == 0 ? v0 : D.v;
        if (!L.relax) {
            // skipped level: v = 0, so the residual is f; restrict it as it is
            pre[l] = nullptr;
            restrict_from(l, f);
            continue;
        }
        const int npl = post_launches(L), prl = pre_launches(L);
        const bool pairs = pairs_on<T>(L.g);
        T *bufs[2] = {((prl + npl) & 1) ? fin : D.w, ((prl + npl) & 1) ? D.w : fin};
        const T *cur = nullptr;
        int nb = 0;
        for (int sw = 0; sw < npre;) {
            if (pairs && npre - sw >= 2) {
                // two sweeps in one launch; the first pair starts from zero (cur == nullptr)
                launch_sweep2<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, cur, bufs[nb], 0);
                sw += 2;
            } else if (sw == 0 && L.g.n0 <= 128 && L.g.N >= ZSWEEP_MIN_CELLS) {
                launch_sweep<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, (const T *)nullptr, bufs[nb], 0);
                sw++;
            } else if (sw == 0) {
                launch_smooth0<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, bufs[nb], 0);
                sw++;
            } else {
                launch_sweep<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, cur, bufs[nb], 0);
                sw++;
            }
            cur = bufs[nb];
            nb ^= 1;
        }
        pre[l] = const_cast<T *>(cur);
        // residual into the level's other buffer (free until post-smoothing), then P^T
        T *rbuf = (cur == fin) ? D.w : fin;
        launch_resid<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, cur, rbuf);
        restrict_from(l, rbuf);
    }
    if (lb < nl) {
        launch_bottom_levels<T>(h, lb);
    } else {
        Level &C = h->lev[nl - 1];
        LevelData<T> &D = data<T>(C);
        coarse_solve<T>(h, nl == 1 ? f0 : D.f, nl == 1 ? v0 : D.v);
    }
    for (int l = top - 1; l >= 0; l--) {
        if (bridged[l]) continue;
        Level &L = h->lev[l];
        LevelData<T> &D = data<T>(L);
        const T *f = l == 0 ? f0 : D.f;
        T *fin = l == 0 ? v0 : D.v;
        if (!L.relax) {
            // skipped level: v = P v_coarse into the level's final buffer
            prolong_to(l, nullptr, fin);
            continue;
        }
        T *cur = pre[l];
        prolong_to(l, cur, cur);
        for (int sw = 0; sw < npost;) {
            T *nxt = (cur == fin) ? D.w : fin;
            if (npost - sw >= 2 && pairs_on<T>(L.g)) {
                launch_sweep2<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, cur, nxt, 1);
                sw += 2;
            } else {
                launch_sweep<T>(s, L.g, D.c, D.a0, D.a1, D.a2, f, cur, nxt, 1);
                sw++;
            }
            cur = nxt;
        }
    }
}

// ---------------------------------------------------------------- graphs

void destroy_graph(ngap_t *h, int prec) {
    if (h->vc_graph[prec]) (void)hipGraphExecDestroy(h->vc_graph[prec]);
    h->vc_graph[prec] = nullptr;
    h->vc_key[prec].clear();
}

void destroy_graphs(ngap_t *h) {
    destroy_graph(h, 0);
    destroy_graph(h, 1);
}

// Everything the recorded V-cycle of one precision depends on: the launch
// sequence follows from the level shapes, coarsening directions, relaxed
// levels, sweep counts and the coarsest solve; the kernel arguments are these
// and the buffer addresses. A setup that leaves all of them as they were
// (a new operator on the same grid and hierarchy) replays the graph it has.
std::vector<long long> cycle_key(const ngap_t *h, int prec) {
    std::vector<long long> k;
    auto P = [&k](const void *p) { k.push_back((long long)(uintptr_t)p); };
    k.insert(k.end(), {(long long)prec, (long long)h->nlev, (long long)h->opts.nu_pre, (long long)h->opts.nu_post,
                       (long long)h->coarse_dense, (long long)h->nc});
    P(h->Ainv);
    P(prec ? (const void *)h->r32 : (const void *)h->r);
    P(prec ? (const void *)h->z32 : (const void *)h->z);
    for (int l = 0; l < h->nlev; l++) {
        const Level &L = h->lev[l];
        k.insert(k.end(), {(long long)L.g.n0, (long long)L.g.n1, (long long)L.g.n2, (long long)L.g.p0,
                           (long long)L.g.p1, (long long)L.g.p2, (long long)L.cdir, (long long)L.relax});
        if (prec) {
            const LevelData<float> &D = L.s;
            for (const void *q : {(const void *)D.c, (const void *)D.a0, (const void *)D.a1, (const void *)D.a2,
                                  (const void *)D.pm, (const void *)D.pp, (const void *)D.f, (const void *)D.v,
                                  (const void *)D.w})
                P(q);
        } else {
            const LevelData<double> &D = L.d;
            for (const void *q : {(const void *)D.c, (const void *)D.a0, (const void *)D.a1, (const void *)D.a2,
                                  (const void *)D.pm, (const void *)D.pp, (const void *)D.f, (const void *)D.v,
                                  (const void *)D.w})
                P(q);
        }
    }
    return k;
}

// Record the V-cycle on the handle's stream (f0 = r / r32, v0 = z / z32).
int capture_vcycle(ngap_t *h, int prec) {
    hipGraph_t g = nullptr;
    HIPCHK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    if (prec)
        vcycle<float>(h, h->r32, h->z32);
    else
        vcycle<double>(h, h->r, h->z);
    hipError_t e = hipStreamEndCapture(h->stream, &g);
    if (e != hipSuccess) {
        g_last_hip = e;
        return NGAP_ERR_HIP;
    }
    e = hipGraphInstantiate(&h->vc_graph[prec], g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) {
        g_last_hip = e;
        h->vc_graph[prec] = nullptr;
        return NGAP_ERR_HIP;
    }
    h->vc_key[prec] = cycle_key(h, prec);
    return 0;
}

// ---------------------------------------------------------------- setup

int do_setup(ngap_t *h, const double *opr, bool on_device, int maxit, double rcvg, int maxlevel,
             const ngap_opts *o) {
    if (!h) return NGAP_ERR_ARG;
    if (!h->init_done) return NGAP_ERR_NOT_INIT;
    if (!opr) return NGAP_ERR_ARG;
    if (h->method != NGAP_PCG_PFMG && h->method != NGAP_GMRES_PFMG) return NGAP_ERR_METHOD;
    if (maxit < 0 || !(rcvg >= 0.0)) return NGAP_ERR_ARG;
    double t0 = now_ms();
    h->setup_done = false;
    ngap_opts op;
    ngap_default_opts(&op);
    if (o) op = *o;
    // 0 = by precision: V(1,1) in FP64 (PFMG's default, as hypre_str leaves it);
    // V(2,2) around the FP32 V-cycle, whose sweeps cost half: 13 iterations
    // instead of 22 at 256^3 (channel), 31.0 against 36.2 ms per solve
    if (op.nu_pre < 1) op.nu_pre = op.precision == NGAP_MIXED ? 2 : 1;
    if (op.nu_post < 1) op.nu_post = op.precision == NGAP_MIXED ? 2 : 1;
    if (op.coarsest_max < 1) op.coarsest_max = 128;
    if (op.skip_relax < 0 || op.skip_relax > 1) return NGAP_ERR_ARG;
    if (op.precision != NGAP_FP64 && op.precision != NGAP_MIXED) return NGAP_ERR_ARG;
    if (h->method == NGAP_GMRES_PFMG && (op.kdim < 1 || op.kdim > 30)) return NGAP_ERR_ARG;
    h->opts = op;
    h->maxit = maxit;
    h->rcvg = rcvg;
    h->maxlevel = maxlevel;
    HIPCHK(hipSetDevice(h->device));
    // tile kernels index with int32 and write one partial per SpMV block;
    // k_level0 indexes the ghosted cells with int32
    if (h->g0.N >= (1LL << 31) || h->nghost >= (1LL << 31)) return NGAP_ERR_UNSUPPORTED;
    {
        int kc;
        if (apply_blocks(h->g0, kc) > MAX_PARTS) return NGAP_ERR_UNSUPPORTED;
    }
    int rc = ensure_base(h);
    if (rc) return rc;
    if (h->method == NGAP_GMRES_PFMG && (h->kdim != op.kdim || !h->gV || !h->gZ)) {
        const size_t N = (size_t)h->g0.N;
        dfree(h, h->gV, sizeof(double) * N * (h->kdim + 1));
        dfree(h, h->gZ, sizeof(double) * N * h->kdim);
        h->gV = h->gZ = nullptr;
        h->kdim = 0;  // set below once both bases exist, so a failed setup never leaves a stale size
        if (dmalloc(h, (void **)&h->gV, sizeof(double) * N * (op.kdim + 1))) return NGAP_ERR_ALLOC;
        if (dmalloc(h, (void **)&h->gZ, sizeof(double) * N * op.kdim)) {
            dfree(h, h->gV, sizeof(double) * N * (op.kdim + 1));
            h->gV = nullptr;
            return NGAP_ERR_ALLOC;
        }
        h->kdim = op.kdim;
    }
    if (h->method == NGAP_GMRES_PFMG) {
        const size_t N = (size_t)h->g0.N;
        if (!h->gm && dmalloc(h, (void **)&h->gm, sizeof(double) * 256)) return NGAP_ERR_ALLOC;
        if (!h->o7 && dmalloc(h, (void **)&h->o7, sizeof(double) * N * 7)) return NGAP_ERR_ALLOC;
        if (!h->h_gm) HIPCHK(hipHostMalloc((void **)&h->h_gm, sizeof(double) * 256, hipHostMallocDefault));
        if (!h->gV || !h->gZ || !h->gm || !h->o7 || !h->h_gm) return NGAP_ERR_ALLOC;
    }
    hipStream_t s = h->stream;
    size_t obytes = sizeof(double) * (size_t)h->nghost * h->nst;
    if (on_device) {
        // the caller's producer may run on another stream: wait for the device
        // first; k_level0 then reads the caller's array and writes the
        // solver's copy of its interior in the same pass
        HIPCHK(hipDeviceSynchronize());
    } else {
        HIPCHK(hipMemcpyAsync(h->opr, opr, obytes, hipMemcpyHostToDevice, s));
    }
    const bool mixed = op.precision == NGAP_MIXED;
    // level 0
    if (h->lev.empty()) {
        h->lev.resize(1);
        h->lev[0].g = h->g0;
        if (alloc_lvl_data(h, h->lev[0].d, h->g0.N, false) || alloc_lvl_data(h, h->lev[0].s, h->g0.N, false))
            return NGAP_ERR_ALLOC;
    }
    Level &L0 = h->lev[0];
    int nb = grid_parts(h->g0.N);
    // level 0 in FP64, and in FP32 for the mixed-precision cycle
    hipLaunchKernelGGL(k_level0, dim3(nb), dim3(NT), 0, s, h->g0, h->gh, h->slots,
                       on_device ? opr : (const double *)h->opr, on_device ? h->opr : (double *)nullptr, L0.d.c,
                       L0.d.a0, L0.d.a1, L0.d.a2, mixed ? L0.s : LevelData<float>{}, h->part, h->parts,
                       h->parts + MAX_PARTS);
    if (h->method == NGAP_GMRES_PFMG)
        hipLaunchKernelGGL(k_soa7, dim3(nb), dim3(NT), 0, s, h->g0, h->gh, h->slots, (const double *)h->opr, h->o7);
    hipLaunchKernelGGL(k_fin_max, dim3(1), dim3(NT), 0, s, (const double *)h->parts, nb, h->scal, (int)S_ASYM);
    hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + MAX_PARTS), nb, h->scal,
                       (int)S_BAD);
    HIPCHK(hipGetLastError());
    // Coarser levels. A setup on a handle whose last setup built a hierarchy
    // with the same options first rebuilds that hierarchy with its coarsening
    // directions, without waiting for the strengths; one read at the end
    // brings every level's strengths, and the directions are checked against
    // them. Levels from the first direction that differs are built again by
    // the loop below, which reads each level's strengths before coarsening it.
    const int nprev = (int)h->lev.size();
    const bool spec = h->spec_valid && nprev >= 2 && h->spec_maxlevel == maxlevel &&
                      h->spec_coarsest == op.coarsest_max;
    h->spec_valid = false;
    int nlev = 1;
    bool have_aniso = false;
    double aniso[2] = {0.0, 0.0};
    if (spec) {
        double *lstr = h->parts + 3 * MAX_PARTS;  // unused by the other setup reductions
        for (int l = 0; l + 1 < nprev; l++) {
            Level &F = h->lev[l];
            Level &C = h->lev[l + 1];
            int np = 0;
            launch_strength(s, F.g, F.d.a0, F.d.a1, F.d.a2, h->parts, &np);
            hipLaunchKernelGGL(k_fin_sums, dim3(1), dim3(NT), 0, s, (const double *)h->parts, np, 3, lstr, 3 * l);
            launch_coarse_build(s, F.g, C.g, F.cdir, F.d.c, F.d.a0, F.d.a1, F.d.a2, C.d.pm, C.d.pp, C.d.c, C.d.a0,
                                C.d.a1, C.d.a2, C.d.f, mixed ? &C.s : nullptr);
        }
        if (op.skip_relax) {
            int np = 0;
            launch_aniso_count(s, L0.g, L0.d.a0, L0.d.a1, L0.d.a2, h->parts, &np);
            hipLaunchKernelGGL(k_fin_sums, dim3(1), dim3(NT), 0, s, (const double *)h->parts, np, 2, lstr,
                               3 * (nprev - 1));
        }
        HIPCHK(hipGetLastError());
        std::vector<double> hs(3 * (size_t)nprev);
        HIPCHK(hipMemcpyAsync(hs.data(), lstr, sizeof(double) * hs.size(), hipMemcpyDeviceToHost, s));
        HIPCHK(hipMemcpyAsync(h->h_scal, h->scal, SCAL_BYTES, hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        h->st.asym = h->h_scal[S_ASYM];
        if (op.check_finite && h->h_scal[S_BAD] > 0.0) return NGAP_ERR_NONFINITE;
        for (int l = 0; l + 1 < nprev; l++) {
            Level &F = h->lev[l];
            for (int d = 0; d < 3; d++) F.str[d] = hs[3 * l + d];
            if (pick_dir(F.g, &hs[3 * l]) != F.cdir) break;
            nlev = l + 2;
        }
        if (op.skip_relax) {
            have_aniso = true;
            aniso[0] = hs[3 * (nprev - 1)];
            aniso[1] = hs[3 * (nprev - 1) + 1];
        }
    } else {
        if ((rc = read_scal(h))) return rc;
        h->st.asym = h->h_scal[S_ASYM];
        if (op.check_finite && h->h_scal[S_BAD] > 0.0) return NGAP_ERR_NONFINITE;
    }
    while (true) {
        Level &F = h->lev[nlev - 1];
        F.cdir = -1;
        if (maxlevel > 0 && nlev >= maxlevel) break;
        if (F.g.N <= op.coarsest_max) break;
        if (nlev >= 64) break;
        int np = 0;
        launch_strength(s, F.g, F.d.a0, F.d.a1, F.d.a2, h->parts, &np);
        hipLaunchKernelGGL(k_fin_sums, dim3(1), dim3(NT), 0, s, (const double *)h->parts, np, 3, h->scal,
                           (int)S_STR0);
        HIPCHK(hipGetLastError());
        if ((rc = read_scal(h))) return rc;
        for (int d = 0; d < 3; d++) F.str[d] = h->h_scal[S_STR0 + d];
        const int best = pick_dir(F.g, F.str);
        if (best < 0) break;
        Geo cg = F.g;
        int per = best == 0 ? F.g.p0 : (best == 1 ? F.g.p1 : F.g.p2);
        int *nd = best == 0 ? &cg.n0 : (best == 1 ? &cg.n1 : &cg.n2);
        *nd = per ? *nd / 2 : (*nd + 1) / 2;
        cg.N = (long long)cg.n0 * cg.n1 * cg.n2;
        F.cdir = best;
        if ((int)h->lev.size() > nlev && h->lev[nlev].g.N != cg.N) {
            for (size_t q = nlev; q < h->lev.size(); q++) free_level(h, h->lev[q]);
            h->lev.resize(nlev);
        }
        if ((int)h->lev.size() == nlev) {
            h->lev.emplace_back();
            Level &C = h->lev.back();
            C.g = cg;
            if (alloc_lvl_data(h, C.d, cg.N, true) || alloc_lvl_data(h, C.s, cg.N, true)) return NGAP_ERR_ALLOC;
        }
        Level &Fr = h->lev[nlev - 1];  // reference may have moved
        Level &C = h->lev[nlev];
        C.g = cg;
        C.cdir = -1;
        launch_coarse_build(s, Fr.g, cg, best, Fr.d.c, Fr.d.a0, Fr.d.a1, Fr.d.a2, C.d.pm, C.d.pp, C.d.c, C.d.a0,
                            C.d.a1, C.d.a2, C.d.f, mixed ? &C.s : nullptr);
        HIPCHK(hipGetLastError());
        nlev++;
    }
    for (size_t q = nlev; q < h->lev.size(); q++) free_level(h, h->lev[q]);
    h->lev.resize(nlev);
    h->nlev = nlev;
    int skip = op.skip_relax;
    h->relax_keep = 1;
    if (skip && nlev > 2) {
        // the skip applies only to a fine level that is locally isotropic
        if (!have_aniso) {
            int np = 0;
            Level &F0 = h->lev[0];
            launch_aniso_count(s, F0.g, F0.d.a0, F0.d.a1, F0.d.a2, h->parts, &np);
            hipLaunchKernelGGL(k_fin_sums, dim3(1), dim3(NT), 0, s, (const double *)h->parts, np, 2, h->scal,
                               (int)S_STR0);
            HIPCHK(hipGetLastError());
            if ((rc = read_scal(h))) return rc;
            aniso[0] = h->h_scal[S_STR0];
            aniso[1] = h->h_scal[S_STR1];
        }
        h->relax_keep = skip_gate(aniso[0], aniso[1]) ? 1 : nlev;
    }
    set_relax(h, skip);
    h->st.skip_relax = skip;
    h->st.relaxed_levels = 0;
    for (int l = 0; l < nlev; l++) h->st.relaxed_levels += h->lev[l].relax ? 1 : 0;
    Level &C = h->lev[nlev - 1];
    h->coarse_dense = C.g.N <= 1024;
    h->coarse_singular = 0;
    if (h->coarse_dense && C.g.N <= COARSE_LDS_MAX) {
        if ((rc = ensure_ainv(h, (int)C.g.N))) return rc;
        launch_coarse_inverse(s, C.g, C.d.c, C.d.a0, C.d.a1, C.d.a2, h->Ainv, h->scal + S_CSING);
        HIPCHK(hipGetLastError());
        if ((rc = read_scal(h))) return rc;
        if (h->h_scal[S_CBAD] > 0.5) return NGAP_ERR_COARSE;
        h->coarse_singular = h->h_scal[S_CSING] > 0.5;
    } else if (h->coarse_dense) {
        if ((rc = build_coarsest_inverse(h))) return rc;
    }
    // (the FP32 copies of the hierarchy for the mixed-precision V-cycle were
    // written by k_level0 and the coarse build)
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s));
    {
        int kc;
        h->apply_parts = apply_blocks(h->lev[0].g, kc);
    }
    // The V-cycle launch sequence is fixed once the hierarchy exists: replay it
    // as a graph, recorded again only when what it recorded has changed. The
    // mixed-precision solve records the FP32 cycle only; its FP64 fallback
    // launches the FP64 cycle directly (or replays a graph still valid).
    for (int prec = 0; prec < 2; prec++) {
        const bool want = op.graphs && (prec == 1 ? mixed : !mixed);
        const bool valid = h->vc_graph[prec] && h->vc_key[prec] == cycle_key(h, prec);
        if (!op.graphs || !valid) destroy_graph(h, prec);
        if (want && !valid && (rc = capture_vcycle(h, prec))) return rc;
    }
    h->setup_done = true;
    h->spec_valid = true;
    h->spec_maxlevel = maxlevel;
    h->spec_coarsest = op.coarsest_max;
    h->st.nlevels = nlev;
    h->st.coarse_singular = h->coarse_singular;
    h->st.setup_ms = now_ms() - t0;
    h->st.cells = h->g0.N;
    h->st.device_bytes = h->dev_bytes;
    return 0;
}

// A device allocation that fails part-way through a setup can leave a level
// or a GMRES basis with some buffers allocated and others null; a later setup
// of the same grid would then reuse the level as it is. So after such a
// failure every device buffer of the handle is released, and the next setup
// allocates all of them again.
int setup_checked(ngap_t *h, const double *opr, bool on_device, int maxit, double rcvg, int maxlevel,
                  const ngap_opts *o) {
    const int rc = do_setup(h, opr, on_device, maxit, rcvg, maxlevel, o);
    if (rc == NGAP_ERR_ALLOC && h) {
        (void)hipSetDevice(h->device);
        (void)hipStreamSynchronize(h->stream);
        free_all(h);
        h->setup_done = false;
    }
    return rc;
}

// ---------------------------------------------------------------- PCG

int exact_residual(ngap_t *h, double *out, int slot) {
    int nb = grid_for(h->g0.N);
    hipLaunchKernelGGL(k_exact_resid, dim3(nb), dim3(NT), 0, h->stream, h->g0, h->gh, h->slots,
                       (const double *)h->opr, (const double *)h->b, (const double *)h->x, out, h->parts);
    hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, h->stream, (const double *)h->parts, nb, h->scal, slot);
    return 0;
}

void precond(ngap_t *h, bool mixed) {
    if (h->vc_graph[mixed ? 1 : 0]) {
        (void)hipGraphLaunch(h->vc_graph[mixed ? 1 : 0], h->stream);
        return;
    }
    if (mixed)
        vcycle<float>(h, h->r32, h->z32);
    else
        vcycle<double>(h, h->r, h->z);
}

int stage_bufs(ngap_t *h) {
    const size_t N = (size_t)h->g0.N;
    if (!h->st_t && dmalloc(h, (void **)&h->st_t, sizeof(double) * N)) return NGAP_ERR_ALLOC;
    if (!h->st_e && dmalloc(h, (void **)&h->st_e, sizeof(double) * N)) return NGAP_ERR_ALLOC;
    return 0;
}

// z = V(r), plus the correction stage z += fn(r - A z) when `stage`. *z64
// tells where the result is: h->z (FP64) or h->z32 (mixed without stage).
int precond_stage(ngap_t *h, bool mixed, bool stage, bool *z64) {
    precond(h, mixed);
    *z64 = !mixed;
    if (!stage) return 0;
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    if (mixed) launch_to_f64(s, N, h->z32, h->z);
    Level &L0 = h->lev[0];
    launch_apply<double>(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, h->z, h->st_t, h->parts + 2 * MAX_PARTS);
    hipLaunchKernelGGL(k_sub_from, dim3(nb), dim3(NT), 0, s, N, (const double *)h->r, h->st_t);
    HIPCHK(hipGetLastError());
    if (h->stage_fn(h->stage_ctx, h->st_t, h->st_e, N, (void *)s)) return NGAP_ERR_STAGE;
    hipLaunchKernelGGL(k_add, dim3(nb), dim3(NT), 0, s, N, h->z, (const double *)h->st_e);
    HIPCHK(hipGetLastError());
    h->st.stage_calls++;
    *z64 = true;
    return 0;
}

// r, z -> rho (restart: p = z)
// p = z + beta p (copy: p = z) with z in FP32 or FP64 and p in the solve's
// direction precision (h->p32)
void launch_update_p(ngap_t *h, bool z64, int copy) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    const double *sc = h->scal;
    float *p32 = reinterpret_cast<float *>(h->p);
    if (h->p32) {
        if (z64)
            hipLaunchKernelGGL((k_update_p<double, float>), dim3(nb), dim3(NT), 0, s, N, p32, (const double *)h->z,
                               sc, copy);
        else
            hipLaunchKernelGGL((k_update_p<float, float>), dim3(nb), dim3(NT), 0, s, N, p32, (const float *)h->z32,
                               sc, copy);
    } else {
        if (z64)
            hipLaunchKernelGGL((k_update_p<double, double>), dim3(nb), dim3(NT), 0, s, N, h->p, (const double *)h->z,
                               sc, copy);
        else
            hipLaunchKernelGGL((k_update_p<float, double>), dim3(nb), dim3(NT), 0, s, N, h->p,
                               (const float *)h->z32, sc, copy);
    }
}

int restart_dir(ngap_t *h, bool mixed, bool first, bool stage) {
    long long N = h->g0.N;
    int nb = grid_for(N);
    bool z64;
    int rc = precond_stage(h, mixed, stage, &z64);
    if (rc) return rc;
    if (!z64)
        hipLaunchKernelGGL(k_dot_rz<float>, dim3(nb), dim3(NT), 0, h->stream, N, (const double *)h->r,
                           (const float *)h->z32, (const double *)nullptr, h->parts, (double *)nullptr);
    else
        hipLaunchKernelGGL(k_dot_rz<double>, dim3(nb), dim3(NT), 0, h->stream, N, (const double *)h->r,
                           (const double *)h->z, (const double *)nullptr, h->parts, (double *)nullptr);
    hipLaunchKernelGGL(k_fin_rho, dim3(1), dim3(NT), 0, h->stream, (const double *)h->parts, nb, h->scal, h->flags,
                       first ? 1 : 0);
    // the mixed solve keeps its directions in FP32 (in the p buffer), the
    // FP64 solve (and a mixed solve fallen back to FP64) in FP64
    h->p32 = mixed;
    launch_update_p(h, z64, 1);
    HIPCHK(hipGetLastError());
    return 0;
}

// Guess stage: x += fn(r), kept only when it lowers the exact residual.
// On entry r = b - A x with ||r||/||b|| = *rel; on exit r and *rel match x.
int guess_stage(ngap_t *h, double bn, double *rel) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    int rc;
    if ((rc = stage_bufs(h))) return rc;
    if (h->stage_fn(h->stage_ctx, h->r, h->st_e, N, (void *)s)) return NGAP_ERR_STAGE;
    h->st.stage_calls++;
    hipLaunchKernelGGL(k_copy, dim3(nb), dim3(NT), 0, s, N, (const double *)h->x, h->q);
    hipLaunchKernelGGL(k_add, dim3(nb), dim3(NT), 0, s, N, h->x, (const double *)h->st_e);
    exact_residual(h, h->r, S_RR);
    HIPCHK(hipGetLastError());
    if ((rc = read_scal(h))) return rc;
    const double rel1 = std::sqrt(h->h_scal[S_RR]) / bn;
    if (rel1 <= *rel) {
        *rel = rel1;
        return 0;
    }
    // rejected (larger or non-finite residual): back to the caller's guess
    hipLaunchKernelGGL(k_copy, dim3(nb), dim3(NT), 0, s, N, (const double *)h->q, h->x);
    exact_residual(h, h->r, S_RR);
    HIPCHK(hipGetLastError());
    if ((rc = read_scal(h))) return rc;
    *rel = std::sqrt(h->h_scal[S_RR]) / bn;
    h->st.fallback |= 2;
    return 0;
}

// p <- z + beta p with z = M r (preconditioner, plus the stage when `stage`):
// r.z (and z.q for the flexible beta), beta, rho, then p
int next_dir(ngap_t *h, bool mixed, bool stage, bool flexible) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    bool z64;
    int rc = precond_stage(h, mixed, stage, &z64);
    if (rc) return rc;
    if (!z64)
        hipLaunchKernelGGL(k_dot_rz<float>, dim3(nb), dim3(NT), 0, s, N, (const double *)h->r, (const float *)h->z32,
                           flexible ? (const double *)h->q : (const double *)nullptr, h->parts,
                           h->parts + MAX_PARTS);
    else
        hipLaunchKernelGGL(k_dot_rz<double>, dim3(nb), dim3(NT), 0, s, N, (const double *)h->r, (const double *)h->z,
                           flexible ? (const double *)h->q : (const double *)nullptr, h->parts,
                           h->parts + MAX_PARTS);
    hipLaunchKernelGGL(k_fin_beta, dim3(1), dim3(NT), 0, s, (const double *)h->parts,
                       (const double *)(h->parts + MAX_PARTS), nb, h->scal, h->flags, flexible ? 1 : 0);
    launch_update_p(h, z64, 0);
    HIPCHK(hipGetLastError());
    return 0;
}

int run_pcg(ngap_t *h) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    bool mixed = h->opts.precision == NGAP_MIXED;
    bool stage_pc = h->stage_fn && (h->stage_flags & NGAP_STAGE_PRECOND) && h->stage_iters > 0;
    // a stage makes the preconditioner vary between iterations: flexible beta
    const bool flexible = mixed || stage_pc;
    int rc;
    h->st.fallback = 0;
    h->st.restarts = 0;
    h->st.stage_calls = 0;
    if (stage_pc && (rc = stage_bufs(h))) return rc;
    hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(64), 0, s, h->flags);
    // from a zero guess (its values and the operator's are known to be finite)
    // the residual is b, and its norm the sum below: the product with the
    // exact operator is left out
    if (h->x_zero)
        hipLaunchKernelGGL(k_copy, dim3(nb), dim3(NT), 0, s, N, (const double *)h->b, h->r);
    else
        exact_residual(h, h->r, S_RR);
    hipLaunchKernelGGL(k_sumsq, dim3(nb), dim3(NT), 0, s, N, (const double *)h->b, h->parts + MAX_PARTS);
    hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + MAX_PARTS), nb, h->scal,
                       (int)S_BB);
    HIPCHK(hipGetLastError());
    if ((rc = read_scal(h))) return rc;
    const double bn = std::sqrt(h->h_scal[S_BB]);
    if (bn == 0.0) {
        hipLaunchKernelGGL(k_zero64, dim3(nb), dim3(NT), 0, s, N, h->x);
        HIPCHK(hipGetLastError());
        h->st.it = 0;
        h->st.rerr = 0.0;
        h->st.true_rerr = 0.0;
        h->st.aerr = 0.0;
        h->st.cnorm_ratio = 0.0;
        h->st.status = NGAP_STATUS_CONVERGED;
        return 0;
    }
    double rel = std::sqrt(h->h_scal[h->x_zero ? S_BB : S_RR]) / bn;
    const double tol = h->rcvg;
    if (h->stage_fn && (h->stage_flags & NGAP_STAGE_GUESS) && rel > tol && std::isfinite(rel)) {
        if ((rc = guess_stage(h, bn, &rel))) return rc;
    }
    int it = 0;
    bool restart = true, first = true, converged = false;
    double tr = rel;
    double q = 1.0;  // last per-iteration reduction of rel
    bool have_q = false;
    double best = rel;  // lowest rel so far, and iterations since it last fell by 10%
    int since_best = 0;
    bool stagnated = false;
    if (mixed) launch_to_f32(s, N, h->r, h->r32);
    while (true) {
        if (rel <= tol) {
            exact_residual(h, h->q, S_RRT);
            HIPCHK(hipGetLastError());
            if ((rc = read_scal(h))) return rc;
            tr = std::sqrt(h->h_scal[S_RRT]) / bn;
            if (tr <= tol || it >= h->maxit) {
                converged = tr <= tol;
                break;
            }
            hipLaunchKernelGGL(k_copy, dim3(nb), dim3(NT), 0, s, N, (const double *)h->q, h->r);
            if (mixed) launch_to_f32(s, N, h->r, h->r32);
            rel = tr;
            restart = true;
            h->st.restarts++;
        }
        if (it >= h->maxit) break;
        if (restart) {
            if ((rc = restart_dir(h, mixed, first, stage_pc && it < h->stage_iters))) return rc;
            first = false;
            restart = false;
        }
        Level &L0 = h->lev[0];
        if (h->p32) {
            const float *p32 = reinterpret_cast<const float *>(h->p);
            launch_apply_x32(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, p32, h->q, h->parts);
            hipLaunchKernelGGL(k_fin_alpha, dim3(1), dim3(NT_FIN), 0, s, (const double *)h->parts, h->apply_parts,
                               h->scal, h->flags);
            hipLaunchKernelGGL(k_update_xr<float>, dim3(nb), dim3(NT), 0, s, N, h->x, h->r, p32,
                               (const double *)h->q, (const double *)h->scal, mixed ? h->r32 : (float *)nullptr,
                               h->parts + MAX_PARTS);
        } else {
            launch_apply<double>(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, h->p, h->q, h->parts);
            hipLaunchKernelGGL(k_fin_alpha, dim3(1), dim3(NT_FIN), 0, s, (const double *)h->parts, h->apply_parts,
                               h->scal, h->flags);
            hipLaunchKernelGGL(k_update_xr<double>, dim3(nb), dim3(NT), 0, s, N, h->x, h->r, (const double *)h->p,
                               (const double *)h->q, (const double *)h->scal, mixed ? h->r32 : (float *)nullptr,
                               h->parts + MAX_PARTS);
        }
        hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + MAX_PARTS), nb, h->scal,
                           (int)S_RR);
        HIPCHK(hipGetLastError());
        it++;
        // Read ||r||^2 and the flags without idling the device: unless this
        // iteration is predicted to be the last, the next direction (V-cycle,
        // r.z, beta, p) is enqueued behind the copy and runs while the host
        // waits for it. That work reads r and writes z, p and the beta/rho
        // scalars only, so when the read then says "converged" or "breakdown"
        // it is discarded: x and r are as without it, and every path that
        // continues from there recomputes p from a fresh preconditioned r.
        const double pred = rel * (have_q ? q : 1.0);
        const bool spec = pred > 4.0 * tol && it < h->maxit;
        HIPCHK(hipMemcpyAsync(h->h_scal, h->scal, SCAL_BYTES, hipMemcpyDeviceToHost, s));
        HIPCHK(hipEventRecord(h->ev_scal, s));
        if (spec && (rc = next_dir(h, mixed, stage_pc && it < h->stage_iters, flexible))) return rc;
        HIPCHK(hipEventSynchronize(h->ev_scal));
        const double rel_prev = rel;
        rel = std::sqrt(h->h_scal[S_RR]) / bn;
        if (rel_prev > 0.0 && std::isfinite(rel)) {
            q = std::min(1.0, rel / rel_prev);
            have_q = true;
        }
        if (h->h_flags[0]) {
            // preconditioner or step breakdown: x, r untouched by a zero step
            hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(64), 0, s, h->flags);
            if (stage_pc) {
                // the stage made the preconditioner indefinite: drop it first
                stage_pc = false;
                h->st.fallback |= 2;
                restart = true;
                continue;
            }
            if (mixed) {
                mixed = false;
                h->st.fallback |= 1;
                restart = true;
                continue;
            }
            if (!std::isfinite(rel)) return NGAP_ERR_BREAKDOWN;
            if (h->st.restarts > 2) return NGAP_ERR_BREAKDOWN;
            h->st.restarts++;
            restart = true;
            continue;
        }
        if (!std::isfinite(rel)) return NGAP_ERR_BREAKDOWN;
        if (rel < 0.9 * best) {
            best = rel;
            since_best = 0;
        } else if (++since_best >= NGAP_STAG_WINDOW && rel > tol) {
            stagnated = true;
            break;
        }
        if (rel <= tol || it >= h->maxit) continue;
        if (!spec && (rc = next_dir(h, mixed, stage_pc && it < h->stage_iters, flexible))) return rc;
    }
    if (!converged && (stagnated || it >= h->maxit) && rel > tol) {
        exact_residual(h, h->q, S_RRT);
        HIPCHK(hipGetLastError());
        if ((rc = read_scal(h))) return rc;
        tr = std::sqrt(h->h_scal[S_RRT]) / bn;
    }
    h->st.it = it;
    h->st.rerr = rel;
    h->st.true_rerr = tr;
    h->st.aerr = tr * bn;
    double rho0 = h->h_scal[S_RHO0], rho = h->h_scal[S_RHO];
    h->st.cnorm_ratio = (rho0 > 0.0 && rho >= 0.0) ? std::sqrt(rho / rho0) : 0.0;
    h->st.status = converged ? NGAP_STATUS_CONVERGED : (stagnated ? NGAP_STATUS_STAGNATED : NGAP_STATUS_MAXIT);
    h->st.precision = mixed ? NGAP_MIXED : NGAP_FP64;
    return 0;
}

// ---------------------------------------------------------------- GMRES

// out[0..nv) = <w, V_i> over the basis in chunks of GB_MAX (device), then
// w -= sum out[i] V_i; with sq_slot >= 0 the squared norm of the updated w
// goes to h->gm[sq_slot]
void cgs_pass(ngap_t *h, double *w, const double *V, int nv, double *out, int sq_slot) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    for (int i0 = 0; i0 < nv; i0 += GB_MAX) {
        const int m = std::min(GB_MAX, nv - i0);
        hipLaunchKernelGGL(k_mdot, dim3(nb), dim3(NT), 0, s, N, (const double *)w, V + (size_t)i0 * N, N, m,
                           h->parts);
        hipLaunchKernelGGL(k_fin_multi, dim3(1), dim3(NT), 0, s, (const double *)h->parts, nb, m, out + i0);
    }
    // classical Gram-Schmidt: every coefficient from the same w, then one update
    for (int i0 = 0; i0 < nv; i0 += GB_MAX) {
        const int m = std::min(GB_MAX, nv - i0);
        const bool last = i0 + m >= nv;
        hipLaunchKernelGGL(k_gs_update, dim3(nb), dim3(NT), 0, s, N, w, V + (size_t)i0 * N, N, m,
                           (const double *)(out + i0), (last && sq_slot >= 0) ? h->parts + 3 * MAX_PARTS : nullptr);
    }
    if (sq_slot >= 0)
        hipLaunchKernelGGL(k_fin_multi, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + 3 * MAX_PARTS), nb, 1,
                           h->gm + sq_slot);
}

// z_j = M^-1 v_j into Z_j: one V-cycle (FP64, or FP32 in mixed precision)
void gmres_precond(ngap_t *h, const double *v, double *zj, bool mixed) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    if (mixed) {
        launch_to_f32(s, N, v, h->r32);
        precond(h, true);
        launch_to_f64(s, N, h->z32, zj);
    } else {
        hipLaunchKernelGGL(k_copy, dim3(nb), dim3(NT), 0, s, N, v, h->r);
        precond(h, false);
        hipLaunchKernelGGL(k_copy, dim3(nb), dim3(NT), 0, s, N, (const double *)h->z, zj);
    }
}

int read_gm(ngap_t *h, int n) {
    HIPCHK(hipMemcpyAsync(h->h_gm, h->gm, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    return 0;
}

// Flexible GMRES(kdim), right-preconditioned (HYPRE's StructGMRES with the
// PFMG preconditioner, hypre_str_class.f90:286-303). Each cycle: v0 = r/|r|;
// per step z_j = M^-1 v_j (one V-cycle of the symmetric part), w = A z_j
// with the exact operator, two passes of classical Gram-Schmidt, Givens
// rotations on the host; then x += Z y. The iteration stops when the
// rotated residual estimate reaches rcvg ||b||, and the true residual
// b - A x, recomputed at each cycle start, confirms it.
int run_gmres(ngap_t *h) {
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipStream_t s = h->stream;
    const bool mixed = h->opts.precision == NGAP_MIXED;
    const int m = h->kdim;
    int rc;
    h->st.fallback = 0;
    h->st.restarts = 0;
    h->st.stage_calls = 0;
    h->st.cnorm_ratio = 0.0;
    h->st.precision = mixed ? NGAP_MIXED : NGAP_FP64;
    hipLaunchKernelGGL(k_sumsq, dim3(nb), dim3(NT), 0, s, N, (const double *)h->b, h->parts + MAX_PARTS);
    hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + MAX_PARTS), nb, h->scal,
                       (int)S_BB);
    HIPCHK(hipGetLastError());
    if ((rc = read_scal(h))) return rc;
    const double bn = std::sqrt(h->h_scal[S_BB]);
    if (bn == 0.0) {
        hipLaunchKernelGGL(k_zero64, dim3(nb), dim3(NT), 0, s, N, h->x);
        HIPCHK(hipGetLastError());
        h->st.it = 0;
        h->st.rerr = h->st.true_rerr = h->st.aerr = 0.0;
        h->st.status = NGAP_STATUS_CONVERGED;
        return 0;
    }
    const double tol = h->rcvg;
    std::vector<double> H((size_t)(m + 1) * m), cs(m), sn(m), g(m + 1), y(m);
    auto Hij = [&](int i, int j) -> double & { return H[(size_t)j * (m + 1) + i]; };
    int it = 0;
    double rel = 0.0, tr = 0.0;
    bool converged = false;
    int cycles = 0;
    while (true) {
        // true residual: r = b - A x into V_0
        hipLaunchKernelGGL(k_apply7, dim3(nb), dim3(NT), 0, s, h->g0, (const double *)h->o7, (const double *)h->b,
                           (const double *)h->x, h->gV, h->parts);
        hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)h->parts, nb, h->scal, (int)S_RRT);
        HIPCHK(hipGetLastError());
        if ((rc = read_scal(h))) return rc;
        const double beta = std::sqrt(h->h_scal[S_RRT]);
        tr = beta / bn;
        if (!std::isfinite(tr)) return NGAP_ERR_BREAKDOWN;
        rel = tr;
        if (tr <= tol) {
            converged = true;
            break;
        }
        if (it >= h->maxit) break;
        if (cycles > 0) h->st.restarts++;
        cycles++;
        hipLaunchKernelGGL(k_scale_to, dim3(nb), dim3(NT), 0, s, N, (const double *)h->gV, 1.0 / beta, h->gV);
        std::fill(g.begin(), g.end(), 0.0);
        g[0] = beta;
        int k = 0;  // columns of this cycle
        for (int j = 0; j < m && it < h->maxit; j++) {
            double *vj = h->gV + (size_t)j * N, *zj = h->gZ + (size_t)j * N;
            double *w = h->gV + (size_t)(j + 1) * N;
            gmres_precond(h, vj, zj, mixed);
            // (no partial sums: as many workgroups as there is work for)
            hipLaunchKernelGGL(k_apply7, dim3(stream_blocks(N, PU)), dim3(NT), 0, s, h->g0, (const double *)h->o7,
                               (const double *)nullptr, (const double *)zj, w, (double *)nullptr);
            cgs_pass(h, w, h->gV, j + 1, h->gm, -1);
            cgs_pass(h, w, h->gV, j + 1, h->gm + 64, 128);
            HIPCHK(hipGetLastError());
            if ((rc = read_gm(h, 129))) return rc;
            for (int i = 0; i <= j; i++) Hij(i, j) = h->h_gm[i] + h->h_gm[64 + i];
            const double hn = std::sqrt(std::max(h->h_gm[128], 0.0));
            Hij(j + 1, j) = hn;
            if (!std::isfinite(hn)) return NGAP_ERR_BREAKDOWN;
            // apply the previous rotations, then a new one zeroing H(j+1, j)
            for (int i = 0; i < j; i++) {
                const double a = Hij(i, j), b = Hij(i + 1, j);
                Hij(i, j) = cs[i] * a + sn[i] * b;
                Hij(i + 1, j) = -sn[i] * a + cs[i] * b;
            }
            const double a = Hij(j, j), b = Hij(j + 1, j);
            const double rr = std::hypot(a, b);
            if (!(rr > 0.0)) return NGAP_ERR_BREAKDOWN;
            cs[j] = a / rr;
            sn[j] = b / rr;
            Hij(j, j) = rr;
            Hij(j + 1, j) = 0.0;
            g[j + 1] = -sn[j] * g[j];
            g[j] = cs[j] * g[j];
            it++;
            k = j + 1;
            rel = std::fabs(g[j + 1]) / bn;
            // converged estimate, or the space is invariant (happy breakdown)
            if (rel <= tol || hn <= 1e-300) break;
            hipLaunchKernelGGL(k_scale_to, dim3(nb), dim3(NT), 0, s, N, (const double *)w, 1.0 / hn, w);
        }
        // y = R^-1 g (upper triangular k x k), x += Z y
        for (int i = k - 1; i >= 0; i--) {
            double t = g[i];
            for (int q = i + 1; q < k; q++) t -= Hij(i, q) * y[q];
            y[i] = t / Hij(i, i);
        }
        for (int i = 0; i < k; i++)
            if (!std::isfinite(y[i])) return NGAP_ERR_BREAKDOWN;
        HIPCHK(hipMemcpyAsync(h->gm + 192, y.data(), sizeof(double) * k, hipMemcpyHostToDevice, s));
        for (int i0 = 0; i0 < k; i0 += GB_MAX) {
            const int mm = std::min(GB_MAX, k - i0);
            hipLaunchKernelGGL(k_lincomb, dim3(nb), dim3(NT), 0, s, N, h->x, (const double *)(h->gZ + (size_t)i0 * N),
                               N, mm, (const double *)(h->gm + 192 + i0));
        }
        HIPCHK(hipGetLastError());
    }
    h->st.it = it;
    h->st.rerr = rel;
    h->st.true_rerr = tr;
    h->st.aerr = tr * bn;
    h->st.status = converged ? NGAP_STATUS_CONVERGED : NGAP_STATUS_MAXIT;
    return 0;
}

__global__ void __launch_bounds__(256) k_zero_fill(double *__restrict__ p, long long n) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) p[i] = 0.0;
}

void free_staging(Staging &S) {
    for (int t = 0; t < STG_THREADS; t++) {
        for (int k = 0; k < 2; k++)
            if (S.ev[t][k]) (void)hipEventDestroy(S.ev[t][k]);
        if (S.st[t]) (void)hipStreamDestroy(S.st[t]);
    }
    if (S.pin) (void)hipHostFree(S.pin);
    S = Staging{};
}

// the pinned chunks, streams and events (once per handle); false: not
// available, the caller copies directly from pageable memory
bool make_staging(Staging &S) {
    if (S.ready) return true;
    bool ok = hipHostMalloc((void **)&S.pin, 2 * STG_THREADS * STG_CHUNK, hipHostMallocDefault) == hipSuccess;
    for (int t = 0; ok && t < STG_THREADS; t++) {
        ok = hipStreamCreateWithFlags(&S.st[t], hipStreamNonBlocking) == hipSuccess;
        for (int k = 0; ok && k < 2; k++)
            ok = hipEventCreateWithFlags(&S.ev[t][k], hipEventDisableTiming) == hipSuccess;
    }
    if (!ok) {
        free_staging(S);
        return false;
    }
    S.ready = true;
    return true;
}

bool all_zero(const double *p, size_t n) {
    // +0.0 and -0.0 both count as zero, as the guess's value is what matters
    for (size_t i = 0; i < n; i++)
        if (p[i] != 0.0) return false;
    return true;
}

// One thread's part of a host -> device copy: bytes from src (pageable) to
// dst (device) through the thread's two pinned chunks. skip_zero: a chunk
// that is all zero is cleared on the device by a fill kernel instead of being
// copied (counted in *zeroed).
int h2d_part(const Staging &S, int t, int device, char *dst, const char *src, size_t bytes, bool skip_zero,
             long long *zeroed) {
    if (hipSetDevice(device) != hipSuccess) return NGAP_ERR_HIP;
    char *pin[2] = {S.pin + (size_t)(2 * t) * STG_CHUNK, S.pin + (size_t)(2 * t + 1) * STG_CHUNK};
    int k = 0;
    for (size_t off = 0; off < bytes; off += STG_CHUNK, k++) {
        const size_t n = std::min(STG_CHUNK, bytes - off);
        const int sl = k & 1;
        if (skip_zero && all_zero((const double *)(src + off), n / sizeof(double))) {
            const long long m = (long long)(n / sizeof(double));
            hipLaunchKernelGGL(k_zero_fill, dim3((unsigned)std::min<long long>((m + 255) / 256, 4096)), dim3(256), 0,
                               S.st[t], (double *)(dst + off), m);
            (*zeroed)++;
            continue;
        }
        // the chunk's previous DMA must have left the pinned buffer
        if (k >= 2 && hipEventSynchronize(S.ev[t][sl]) != hipSuccess) return NGAP_ERR_HIP;
        std::memcpy(pin[sl], src + off, n);
        if (hipMemcpyAsync(dst + off, pin[sl], n, hipMemcpyHostToDevice, S.st[t]) != hipSuccess ||
            hipEventRecord(S.ev[t][sl], S.st[t]) != hipSuccess)
            return NGAP_ERR_HIP;
    }
    if (hipGetLastError() != hipSuccess) return NGAP_ERR_HIP;
    return hipStreamSynchronize(S.st[t]) == hipSuccess ? 0 : NGAP_ERR_HIP;
}

// One thread's part of a device -> host copy: the DMA of chunk k+1 runs while
// chunk k is copied from pinned to pageable memory.
int d2h_part(const Staging &S, int t, int device, char *dst, const char *src, size_t bytes) {
    if (hipSetDevice(device) != hipSuccess) return NGAP_ERR_HIP;
    char *pin[2] = {S.pin + (size_t)(2 * t) * STG_CHUNK, S.pin + (size_t)(2 * t + 1) * STG_CHUNK};
    const size_t nch = (bytes + STG_CHUNK - 1) / STG_CHUNK;
    auto issue = [&](size_t k) {
        const size_t off = k * STG_CHUNK, n = std::min(STG_CHUNK, bytes - off);
        return hipMemcpyAsync(pin[k & 1], src + off, n, hipMemcpyDeviceToHost, S.st[t]) == hipSuccess &&
               hipEventRecord(S.ev[t][k & 1], S.st[t]) == hipSuccess;
    };
    if (nch > 0 && !issue(0)) return NGAP_ERR_HIP;
    for (size_t k = 0; k < nch; k++) {
        if (k + 1 < nch && !issue(k + 1)) return NGAP_ERR_HIP;
        if (hipEventSynchronize(S.ev[t][k & 1]) != hipSuccess) return NGAP_ERR_HIP;
        const size_t off = k * STG_CHUNK, n = std::min(STG_CHUNK, bytes - off);
        std::memcpy(dst + off, pin[k & 1], n);
    }
    return 0;
}

// Copy `bytes` (a multiple of 8) between the caller's pageable array and a
// device array on STG_THREADS threads; parts are contiguous and 8-byte
// aligned. A thread that cannot be started runs its part on the caller's
// thread. The device array is complete (H2D) or the host array written (D2H)
// when this returns 0.
int staged_copy(ngap_t *h, bool to_device, char *dev, char *host, size_t bytes, bool skip_zero) {
    Staging &S = h->stg;
    const size_t words = bytes / sizeof(double);
    int rcs[STG_THREADS] = {};
    long long zs[STG_THREADS] = {};
    auto part = [&](int t) {
        const size_t w0 = words * (size_t)t / STG_THREADS, w1 = words * (size_t)(t + 1) / STG_THREADS;
        const size_t o = w0 * sizeof(double), n = (w1 - w0) * sizeof(double);
        rcs[t] = to_device ? h2d_part(S, t, h->device, dev + o, host + o, n, skip_zero, &zs[t])
                           : d2h_part(S, t, h->device, host + o, dev + o, n);
    };
    std::vector<std::thread> th;
    std::vector<int> inline_parts;
    for (int t = 1; t < STG_THREADS; t++) {
        try {
            th.emplace_back(part, t);
        } catch (...) {
            inline_parts.push_back(t);
        }
    }
    part(0);
    for (int t : inline_parts) part(t);
    for (auto &x : th) x.join();
    h->zero_chunks = 0;
    for (int t = 0; t < STG_THREADS; t++) {
        if (rcs[t]) return rcs[t];
        h->zero_chunks += zs[t];
    }
    return hipSetDevice(h->device) == hipSuccess ? 0 : NGAP_ERR_HIP;
}

int do_solve(ngap_t *h, const double *rhs, double *sol, bool on_device, int *it, double *rerr, double *aerr) {
    if (!h || !rhs || !sol) return NGAP_ERR_ARG;
    if (!h->setup_done) return NGAP_ERR_NOT_SETUP;
    double t0 = now_ms();
    HIPCHK(hipSetDevice(h->device));
    hipStream_t s = h->stream;
    const double *drhs = rhs;
    double *dsol = sol;
    double tc = 0.0;
    size_t gb = sizeof(double) * (size_t)h->nghost;
    if (on_device) {
        // rhs/sol may have been written on another stream: wait for the device first
        HIPCHK(hipDeviceSynchronize());
    } else {
        double c0 = now_ms();
        if (make_staging(h->stg)) {
            // the previous solve's work on the handle's stream may still read rhs_g / sol_g
            HIPCHK(hipStreamSynchronize(s));
            int rc = staged_copy(h, true, (char *)h->rhs_g, (char *)rhs, gb, false);
            if (!rc) rc = staged_copy(h, true, (char *)h->sol_g, (char *)sol, gb, true);
            if (rc) return rc;
        } else {
            HIPCHK(hipMemcpyAsync(h->rhs_g, rhs, gb, hipMemcpyHostToDevice, s));
            HIPCHK(hipMemcpyAsync(h->sol_g, sol, gb, hipMemcpyHostToDevice, s));
            HIPCHK(hipStreamSynchronize(s));
        }
        tc += now_ms() - c0;
        drhs = h->rhs_g;
        dsol = h->sol_g;
    }
    const long long N = h->g0.N;
    // counts are exact in any order, so these take more partial sums than the
    // solver's reductions (256^3: 100 us with 1024 workgroups, 66 us now)
    const int nb = std::min(grid_parts(N), 4096);
    hipLaunchKernelGGL(k_gather, dim3(nb), dim3(NT), 0, s, h->g0, h->gh, drhs, (const unsigned char *)h->part, h->b,
                       h->opts.check_finite ? h->parts : (double *)nullptr, (double *)nullptr);
    if (h->opts.check_finite)
        hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)h->parts, nb, h->scal, (int)S_BAD);
    hipLaunchKernelGGL(k_gather, dim3(nb), dim3(NT), 0, s, h->g0, h->gh, (const double *)dsol,
                       (const unsigned char *)h->part, h->x, h->opts.check_finite ? h->parts + MAX_PARTS : nullptr,
                       h->opts.check_finite ? h->parts + 2 * MAX_PARTS : nullptr);
    h->x_zero = false;
    if (h->opts.check_finite) {
        hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + MAX_PARTS), nb, h->scal,
                           (int)S_RRT);
        hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, s, (const double *)(h->parts + 2 * MAX_PARTS), nb, h->scal,
                           (int)S_XNZ);
        HIPCHK(hipGetLastError());
        int rc = read_scal(h);
        if (rc) return rc;
        if (h->h_scal[S_BAD] > 0.0 || h->h_scal[S_RRT] > 0.0) return NGAP_ERR_NONFINITE;
        h->x_zero = h->h_scal[S_XNZ] == 0.0;
    }
    HIPCHK(hipGetLastError());
    int rc = h->method == NGAP_GMRES_PFMG ? run_gmres(h) : run_pcg(h);
    if (rc) return rc;
    hipLaunchKernelGGL(k_scatter, dim3(stream_blocks(N, 4)), dim3(NT), 0, s, h->g0, h->gh, (const double *)h->x, dsol);
    HIPCHK(hipGetLastError());
    if (!on_device) {
        HIPCHK(hipStreamSynchronize(s));
        double c0 = now_ms();
        if (h->stg.ready) {
            int rc = staged_copy(h, false, (char *)h->sol_g, (char *)sol, gb, false);
            if (rc) return rc;
        } else {
            HIPCHK(hipMemcpyAsync(sol, h->sol_g, gb, hipMemcpyDeviceToHost, s));
            HIPCHK(hipStreamSynchronize(s));
        }
        tc += now_ms() - c0;
    } else {
        HIPCHK(hipStreamSynchronize(s));
    }
    h->st.copy_ms = tc;
    h->st.solve_ms = now_ms() - t0;
    if (it) *it = h->st.it;
    if (rerr) *rerr = h->st.rerr;
    if (aerr) *aerr = h->st.aerr;
    if (h->opts.verbose > 0)
        std::fprintf(stderr, "[ngap] it=%d rerr=%.3e true=%.3e levels=%d %s%s solve=%.3f ms\n", h->st.it,
                     h->st.rerr, h->st.true_rerr, h->st.nlevels, h->st.precision == NGAP_MIXED ? "mixed" : "fp64",
                     h->st.fallback ? " (fallback)" : "", h->st.solve_ms);
    return 0;
}

// Device staging for the test hooks
struct Tmp {
    std::vector<std::pair<void *, size_t>> v;
    ~Tmp() {
        for (auto &q : v) (void)hipFree(q.first);
    }
    template <typename T>
    T *get(size_t n) {
        void *p = nullptr;
        if (hipMalloc(&p, sizeof(T) * (n ? n : 1)) != hipSuccess) return nullptr;
        v.push_back({p, sizeof(T) * n});
        return (T *)p;
    }
};

template <typename T>
int up(hipStream_t s, Tmp &tmp, const double *src, size_t n, T **out) {
    double *d = tmp.get<double>(n);
    if (!d) return NGAP_ERR_ALLOC;
    HIPCHK(hipMemcpyAsync(d, src, sizeof(double) * n, hipMemcpyHostToDevice, s));
    if constexpr (std::is_same<T, double>::value) {
        *out = d;
    } else {
        float *f = tmp.get<float>(n);
        if (!f) return NGAP_ERR_ALLOC;
        launch_to_f32(s, (long long)n, d, f);
        *out = f;
    }
    return 0;
}

template <typename T>
int down(hipStream_t s, Tmp &tmp, const T *src, size_t n, double *dst) {
    const double *d;
    if constexpr (std::is_same<T, double>::value) {
        d = src;
    } else {
        double *t = tmp.get<double>(n);
        if (!t) return NGAP_ERR_ALLOC;
        launch_to_f64(s, (long long)n, src, t);
        d = t;
    }
    HIPCHK(hipMemcpyAsync(dst, d, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    return 0;
}

}  // namespace

namespace {

template <typename T>
static int t_apply(ngap_t *h, int l, const double *x, double *y) {
    Tmp tmp;
    Level &L = h->lev[l];
    LevelData<T> &D = data<T>(L);
    size_t n = (size_t)L.g.N;
    T *dx, *dy = tmp.get<T>(n);
    int rc = up<T>(h->stream, tmp, x, n, &dx);
    if (rc || !dy) return rc ? rc : NGAP_ERR_ALLOC;
    launch_apply<T>(h->stream, L.g, D.c, D.a0, D.a1, D.a2, dx, dy, nullptr);
    HIPCHK(hipGetLastError());
    return down<T>(h->stream, tmp, dy, n, y);
}

template <typename T>
static int t_rbgs(ngap_t *h, int l, const double *f, double *v, int order) {
    Tmp tmp;
    Level &L = h->lev[l];
    LevelData<T> &D = data<T>(L);
    size_t n = (size_t)L.g.N;
    T *df, *dv, *dout = tmp.get<T>(n);
    int rc = up<T>(h->stream, tmp, f, n, &df);
    if (!rc) rc = up<T>(h->stream, tmp, v, n, &dv);
    if (rc || !dout) return rc ? rc : NGAP_ERR_ALLOC;
    if ((order & 6) == 6)  // the first two sweeps from a zero iterate in one launch
        launch_sweep2<T>(h->stream, L.g, D.c, D.a0, D.a1, D.a2, df, (const T *)nullptr, dout, order & 1,
                         (order & 8) != 0);
    else if (order & 2)  // first sweep from a zero iterate (the V-cycle's pre-smoothing)
        launch_smooth0<T>(h->stream, L.g, D.c, D.a0, D.a1, D.a2, df, dout, order & 1);
    else if (order & 4)  // two sweeps of the same order in one launch (the post-smoothing pair)
        launch_sweep2<T>(h->stream, L.g, D.c, D.a0, D.a1, D.a2, df, dv, dout, order & 1, (order & 8) != 0);
    else  // bit 3: the 64-wide tiles (pairs: one cell per lane) on every level; bit 4: the single sweep from a zero iterate
        launch_sweep<T>(h->stream, L.g, D.c, D.a0, D.a1, D.a2, df, (order & 16) ? (const T *)nullptr : dv, dout,
                        order & 1, (order & 8) != 0);
    HIPCHK(hipGetLastError());
    return down<T>(h->stream, tmp, dout, n, v);
}

template <typename T>
static int t_rr(ngap_t *h, int l, const double *f, const double *v, double *fc, bool vec) {
    Tmp tmp;
    Level &L = h->lev[l];
    Level &C = h->lev[l + 1];
    LevelData<T> &D = data<T>(L);
    LevelData<T> &DC = data<T>(C);
    size_t n = (size_t)L.g.N, nc = (size_t)C.g.N;
    T *df, *dv, *dr = tmp.get<T>(n), *dfc = tmp.get<T>(nc);
    int rc = up<T>(h->stream, tmp, f, n, &df);
    if (!rc) rc = up<T>(h->stream, tmp, v, n, &dv);
    if (rc || !dfc || !dr) return rc ? rc : NGAP_ERR_ALLOC;
    launch_resid<T>(h->stream, L.g, D.c, D.a0, D.a1, D.a2, df, dv, dr);
    launch_gather<T>(h->stream, L.g, C.g, L.cdir, dr, DC.pm, DC.pp, dfc, vec);
    HIPCHK(hipGetLastError());
    return down<T>(h->stream, tmp, dfc, nc, fc);
}

template <typename T>
static int t_pr(ngap_t *h, int l, const double *vc, double *v, bool vec) {
    Tmp tmp;
    Level &L = h->lev[l];
    Level &C = h->lev[l + 1];
    LevelData<T> &DC = data<T>(C);
    size_t n = (size_t)L.g.N, nc = (size_t)C.g.N;
    T *dvc, *dv;
    int rc = up<T>(h->stream, tmp, vc, nc, &dvc);
    if (!rc) rc = up<T>(h->stream, tmp, v, n, &dv);
    if (rc) return rc;
    launch_prolong_to<T>(h->stream, L.g, C.g, L.cdir, DC.pm, DC.pp, dvc, dv, dv, vec);
    HIPCHK(hipGetLastError());
    return down<T>(h->stream, tmp, dv, n, v);
}

template <typename T>
static int t_cs(ngap_t *h, const double *f, double *v) {
    Tmp tmp;
    Level &C = h->lev[h->nlev - 1];
    size_t n = (size_t)C.g.N;
    T *df, *dv = tmp.get<T>(n);
    int rc = up<T>(h->stream, tmp, f, n, &df);
    if (rc || !dv) return rc ? rc : NGAP_ERR_ALLOC;
    coarse_solve<T>(h, df, dv);
    HIPCHK(hipGetLastError());
    return down<T>(h->stream, tmp, dv, n, v);
}

template <typename T>
static int t_vc(ngap_t *h, const double *r, double *z) {
    Tmp tmp;
    size_t n = (size_t)h->g0.N;
    T *dr, *dz = tmp.get<T>(n);
    int rc = up<T>(h->stream, tmp, r, n, &dr);
    if (rc || !dz) return rc ? rc : NGAP_ERR_ALLOC;
    vcycle<T>(h, dr, dz);
    HIPCHK(hipGetLastError());
    return down<T>(h->stream, tmp, dz, n, z);
}

}  // namespace

// ====================================================================== C ABI

extern "C" {

int ngap_default_opts(ngap_opts *o) {
    if (!o) return NGAP_ERR_ARG;
    o->precision = NGAP_FP64;
    o->nu_pre = 0;
    o->nu_post = 0;
    o->coarsest_max = 128;
    o->check_finite = 1;
    o->verbose = 0;
    o->graphs = 1;
    o->kdim = 5;
    o->skip_relax = 1;
    return 0;
}

const char *ngap_strerror(int code) {
    switch (code) {
        case NGAP_OK: return "ok";
        case NGAP_ERR_ARG: return "invalid argument";
        case NGAP_ERR_STENCIL: return "stencil is not the 7-point set";
        case NGAP_ERR_NOT_INIT: return "solver has not been initialised";
        case NGAP_ERR_NOT_SETUP: return "solver has not been setup";
        case NGAP_ERR_METHOD: return "unknown or unsupported solution method";
        case NGAP_ERR_UNSUPPORTED: return "grid not supported (PCG: periodic direction with an odd number of cells; fourier3d: non-periodic direction)";
        case NGAP_ERR_NOT_CIRCULANT: return "operator must be uniform in space";
        case NGAP_ERR_SINGULAR: return "transformed operator has elements near zero or NaN";
        case NGAP_ERR_HIP: return "HIP runtime error";
        case NGAP_ERR_NONFINITE: return "non-finite value in opr, rhs or initial guess";
        case NGAP_ERR_BREAKDOWN: return "PCG breakdown";
        case NGAP_ERR_ALLOC: return "allocation failed";
        case NGAP_ERR_COARSE: return "coarsest-level factorisation failed";
        case NGAP_ERR_STAGE: return "correction stage failed";
        default: return "unknown error";
    }
}

int ngap_create(ngap_t **hp, const ngap_grid *g, int nst, const int *stc, int method) {
    if (!hp) return NGAP_ERR_ARG;
    *hp = nullptr;
    if (!g || !stc || nst < 1) return NGAP_ERR_ARG;
    if (g->nx < 1 || g->ny < 1 || g->nz < 1) return NGAP_ERR_ARG;
    // one GPU holds the whole grid: local bounds must span the global grid
    if (g->imax_ - g->imin_ + 1 != g->nx || g->jmax_ - g->jmin_ + 1 != g->ny || g->kmax_ - g->kmin_ + 1 != g->nz)
        return NGAP_ERR_ARG;
    if (g->imino_ > g->imin_ || g->imaxo_ < g->imax_ || g->jmino_ > g->jmin_ || g->jmaxo_ < g->jmax_ ||
        g->kmino_ > g->kmin_ || g->kmaxo_ < g->kmax_)
        return NGAP_ERR_ARG;
    ngap_t *h = new (std::nothrow) ngap_t();
    if (!h) return NGAP_ERR_ALLOC;
    h->g = *g;
    h->nst = nst;
    h->stc.assign(stc, stc + 3 * nst);
    h->method = method;
    h->st.it = 0;
    ngap_default_opts(&h->opts);
    *hp = h;
    return 0;
}

int ngap_init(ngap_t *h) {
    if (!h) return NGAP_ERR_ARG;
    // inverse stencil map (hypre_str_class.f90:116-123): slot of each 7-point offset
    const int want[7][3] = {{0, 0, 0}, {1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}};
    if (h->nst != 7) return NGAP_ERR_STENCIL;
    for (int w = 0; w < 7; w++) {
        int found = -1;
        for (int st = 0; st < h->nst; st++) {
            int dx = h->stc[st], dy = h->stc[h->nst + st], dz = h->stc[2 * h->nst + st];
            if (dx == want[w][0] && dy == want[w][1] && dz == want[w][2]) {
                if (found >= 0) return NGAP_ERR_STENCIL;
                found = st;
            }
        }
        if (found < 0) return NGAP_ERR_STENCIL;
        h->slots.s[w] = found;
    }
    h->slots.nst = h->nst;
    const ngap_grid &g = h->g;
    const int n3[3] = {g.nx, g.ny, g.nz}, p3[3] = {g.xper != 0, g.yper != 0, g.zper != 0};
    for (int d = 0; d < 3; d++)
        if (p3[d] && n3[d] >= 3 && (n3[d] & 1)) return NGAP_ERR_UNSUPPORTED;
    h->g0.n0 = g.nx;
    h->g0.n1 = g.ny;
    h->g0.n2 = g.nz;
    h->g0.p0 = p3[0];
    h->g0.p1 = p3[1];
    h->g0.p2 = p3[2];
    h->g0.N = (long long)g.nx * g.ny * g.nz;
    h->gh.nxo = g.imaxo_ - g.imino_ + 1;
    h->gh.nyo = g.jmaxo_ - g.jmino_ + 1;
    long long nzo = g.kmaxo_ - g.kmino_ + 1;
    h->gh.oi = g.imin_ - g.imino_;
    h->gh.oj = g.jmin_ - g.jmino_;
    h->gh.ok = g.kmin_ - g.kmino_;
    h->nghost = h->gh.nxo * h->gh.nyo * nzo;
    if (!h->init_done) {
        if (hipGetDevice(&h->device) != hipSuccess) return NGAP_ERR_HIP;
        if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) return NGAP_ERR_HIP;
        if (hipEventCreateWithFlags(&h->ev_scal, hipEventDisableTiming) != hipSuccess) return NGAP_ERR_HIP;
    }
    h->init_done = true;
    return 0;
}

int ngap_setup(ngap_t *h, const double *opr, int maxit, double rcvg, int maxlevel, const ngap_opts *o) {
    return setup_checked(h, opr, false, maxit, rcvg, maxlevel, o);
}

int ngap_setup_device(ngap_t *h, const double *d_opr, int maxit, double rcvg, int maxlevel, const ngap_opts *o) {
    return setup_checked(h, d_opr, true, maxit, rcvg, maxlevel, o);
}

int ngap_solve(ngap_t *h, const double *rhs, double *sol, int *it, double *rerr, double *aerr) {
    return do_solve(h, rhs, sol, false, it, rerr, aerr);
}

int ngap_solve_device(ngap_t *h, const double *d_rhs, double *d_sol, int *it, double *rerr, double *aerr) {
    return do_solve(h, d_rhs, d_sol, true, it, rerr, aerr);
}

int ngap_residual_device(ngap_t *h, const double *d_rhs, const double *d_sol, double *d_res, double *rnorm) {
    if (!h || !d_rhs || !d_sol || !d_res) return NGAP_ERR_ARG;
    if (!h->setup_done) return NGAP_ERR_NOT_SETUP;
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipDeviceSynchronize());
    hipStream_t s = h->stream;
    const long long N = h->g0.N;
    const int nb = grid_for(N);
    hipLaunchKernelGGL(k_gather, dim3(nb), dim3(NT), 0, s, h->g0, h->gh, d_rhs, (const unsigned char *)h->part, h->b,
                       (double *)nullptr, (double *)nullptr);
    hipLaunchKernelGGL(k_gather, dim3(nb), dim3(NT), 0, s, h->g0, h->gh, d_sol, (const unsigned char *)h->part, h->x,
                       (double *)nullptr, (double *)nullptr);
    exact_residual(h, d_res, S_RRT);
    HIPCHK(hipGetLastError());
    int rc = read_scal(h);
    if (rc) return rc;
    if (rnorm) *rnorm = std::sqrt(h->h_scal[S_RRT]);
    return 0;
}

int ngap_apply_device(ngap_t *h, const double *d_x, double *d_y) {
    if (!h || !d_x || !d_y) return NGAP_ERR_ARG;
    if (!h->setup_done) return NGAP_ERR_NOT_SETUP;
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipDeviceSynchronize());
    Level &L0 = h->lev[0];
    launch_apply<double>(h->stream, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, d_x, d_y, h->parts + 2 * MAX_PARTS);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(h->stream));
    return 0;
}

int ngap_set_stage(ngap_t *h, ngap_stage_fn fn, void *ctx, int flags, int precond_iters) {
    if (!h || precond_iters < 0 || (flags & ~(NGAP_STAGE_GUESS | NGAP_STAGE_PRECOND))) return NGAP_ERR_ARG;
    h->stage_fn = fn;
    h->stage_ctx = fn ? ctx : nullptr;
    h->stage_flags = fn ? flags : 0;
    h->stage_iters = fn ? precond_iters : 0;
    return 0;
}

int ngap_set_tolerance(ngap_t *h, int maxit, double rcvg) {
    if (!h || maxit < 0 || !(rcvg >= 0.0)) return NGAP_ERR_ARG;
    h->maxit = maxit;
    h->rcvg = rcvg;
    return 0;
}

int ngap_destroy(ngap_t *h) {
    if (!h) return NGAP_ERR_ARG;
    if (h->init_done) {
        (void)hipSetDevice(h->device);
        if (h->stream) (void)hipStreamSynchronize(h->stream);
        free_all(h);
        if (h->h_scal) (void)hipHostFree(h->h_scal);
        if (h->h_gm) (void)hipHostFree(h->h_gm);
        free_staging(h->stg);
        if (h->ev_scal) (void)hipEventDestroy(h->ev_scal);
        if (h->stream) (void)hipStreamDestroy(h->stream);
    }
    delete h;
    return 0;
}

int ngap_last_stats(const ngap_t *h, ngap_stats *s) {
    if (!h || !s) return NGAP_ERR_ARG;
    *s = h->st;
    s->device_bytes = h->dev_bytes;
    return 0;
}

// ------------------------------------------------------------ test hooks

int ngapt_nlevels(const ngap_t *h) { return (h && h->setup_done) ? h->nlev : -1; }

int ngapt_pairs(const int *n3, const int *per3, int prec) {
    if (!n3 || !per3) return -1;
    Geo g{};
    g.n0 = n3[0], g.n1 = n3[1], g.n2 = n3[2];
    g.p0 = per3[0], g.p1 = per3[1], g.p2 = per3[2];
    g.N = (long long)g.n0 * g.n1 * g.n2;
    if (!(prec ? pairs_on<float>(g) : pairs_on<double>(g))) return 0;
    return (prec ? pair_form<float>(g) : pair_form<double>(g)) ? 2 : 1;
}

int ngapt_fail_alloc(ngap_t *h, int n) {
    if (!h || n < 0) return NGAP_ERR_ARG;
    h->fail_alloc = n;
    return 0;
}

int ngapt_level_info(const ngap_t *h, int l, int *dims3, int *cdir) {
    if (!h || !h->setup_done || l < 0 || l >= h->nlev || !dims3 || !cdir) return NGAP_ERR_ARG;
    dims3[0] = h->lev[l].g.n0;
    dims3[1] = h->lev[l].g.n1;
    dims3[2] = h->lev[l].g.n2;
    *cdir = h->lev[l].cdir;
    return 0;
}

int ngapt_level_coefs(const ngap_t *h, int l, double *c, double *ax, double *ay, double *az, double *pm, double *pp) {
    if (!h || !h->setup_done || l < 0 || l >= h->nlev) return NGAP_ERR_ARG;
    const Level &L = h->lev[l];
    size_t b = sizeof(double) * (size_t)L.g.N;
    if (c) HIPCHK(hipMemcpy(c, L.d.c, b, hipMemcpyDeviceToHost));
    if (ax) HIPCHK(hipMemcpy(ax, L.d.a0, b, hipMemcpyDeviceToHost));
    if (ay) HIPCHK(hipMemcpy(ay, L.d.a1, b, hipMemcpyDeviceToHost));
    if (az) HIPCHK(hipMemcpy(az, L.d.a2, b, hipMemcpyDeviceToHost));
    if (l > 0) {
        if (pm) HIPCHK(hipMemcpy(pm, L.d.pm, b, hipMemcpyDeviceToHost));
        if (pp) HIPCHK(hipMemcpy(pp, L.d.pp, b, hipMemcpyDeviceToHost));
    } else {
        if (pm) std::memset(pm, 0, b);
        if (pp) std::memset(pp, 0, b);
    }
    return 0;
}

#define TEST_GUARD(l)                                                                   \
    if (!h || !h->setup_done || (l) < 0 || (l) >= h->nlev) return NGAP_ERR_ARG;        \
    if (prec == 1 && h->opts.precision != NGAP_MIXED) return NGAP_ERR_ARG;              \
    if (prec != 0 && prec != 1) return NGAP_ERR_ARG;                                    \
    HIPCHK(hipSetDevice(h->device));

int ngapt_apply(ngap_t *h, int l, int prec, const double *x, double *y) {
    TEST_GUARD(l);
    return prec ? t_apply<float>(h, l, x, y) : t_apply<double>(h, l, x, y);
}

int ngapt_rbgs(ngap_t *h, int l, int prec, const double *f, double *v, int order) {
    TEST_GUARD(l);
    return prec ? t_rbgs<float>(h, l, f, v, order) : t_rbgs<double>(h, l, f, v, order);
}

int ngapt_resid_restrict(ngap_t *h, int l, int prec, const double *f, const double *v, double *fc) {
    const bool vec = !(prec & 2);
    prec &= ~2;
    TEST_GUARD(l + 1);
    return prec ? t_rr<float>(h, l, f, v, fc, vec) : t_rr<double>(h, l, f, v, fc, vec);
}

int ngapt_prolong_add(ngap_t *h, int l, int prec, const double *vc, double *v) {
    const bool vec = !(prec & 2);
    prec &= ~2;
    TEST_GUARD(l + 1);
    return prec ? t_pr<float>(h, l, vc, v, vec) : t_pr<double>(h, l, vc, v, vec);
}

int ngapt_coarse_solve(ngap_t *h, int prec, const double *f, double *v) {
    TEST_GUARD(0);
    return prec ? t_cs<float>(h, f, v) : t_cs<double>(h, f, v);
}

int ngapt_vcycle(ngap_t *h, int prec, const double *r, double *z) {
    TEST_GUARD(0);
    return prec ? t_vc<float>(h, r, z) : t_vc<double>(h, r, z);
}

int ngapt_apply_exact(ngap_t *h, const double *x, double *y) {
    if (!h || !h->setup_done || !x || !y) return NGAP_ERR_ARG;
    HIPCHK(hipSetDevice(h->device));
    size_t n = (size_t)h->g0.N;
    // y = A x  computed as b - (b - A x) with b = 0 in the q buffer
    hipLaunchKernelGGL(k_zero64, dim3(grid_for(n)), dim3(NT), 0, h->stream, (long long)n, h->b);
    HIPCHK(hipMemcpyAsync(h->x, x, sizeof(double) * n, hipMemcpyHostToDevice, h->stream));
    exact_residual(h, h->q, S_RRT);
    HIPCHK(hipGetLastError());
    std::vector<double> t(n);
    HIPCHK(hipMemcpyAsync(t.data(), h->q, sizeof(double) * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    for (size_t i = 0; i < n; i++) y[i] = -t[i];
    return 0;
}

int ngapt_dot(ngap_t *h, long long n, const double *x, const double *y, double *out) {
    if (!h || !h->setup_done || n < 0 || !x || !y || !out) return NGAP_ERR_ARG;
    HIPCHK(hipSetDevice(h->device));
    Tmp tmp;
    double *dx = tmp.get<double>(n), *dy = tmp.get<double>(n);
    if (!dx || !dy) return NGAP_ERR_ALLOC;
    HIPCHK(hipMemcpyAsync(dx, x, sizeof(double) * n, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(dy, y, sizeof(double) * n, hipMemcpyHostToDevice, h->stream));
    int nb = grid_for(n);
    hipLaunchKernelGGL((k_dot<double, double>), dim3(nb), dim3(NT), 0, h->stream, n, (const double *)dx,
                       (const double *)dy, h->parts);
    hipLaunchKernelGGL(k_fin_sum, dim3(1), dim3(NT), 0, h->stream, (const double *)h->parts, nb, h->scal, (int)S_RRT);
    HIPCHK(hipGetLastError());
    int rc = read_scal(h);
    if (rc) return rc;
    *out = h->h_scal[S_RRT];
    return 0;
}

int ngapt_time_kernel(ngap_t *h, int kid, int prec, int reps, double *avg_ms, double *bytes) {
    TEST_GUARD(0);
    if (reps < 1 || !avg_ms || !bytes) return NGAP_ERR_ARG;
    hipStream_t s = h->stream;
    Level &L0 = h->lev[0];
    const long long N = L0.g.N;
    const double w = prec ? 4.0 : 8.0;
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    auto launch = [&]() -> int {
        switch (kid) {
            case NGAPT_K_SPMV:
                if (prec)
                    launch_apply<float>(s, L0.g, L0.s.c, L0.s.a0, L0.s.a1, L0.s.a2, h->z32, h->r32, nullptr);
                else
                    launch_apply<double>(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, h->p, h->q, h->parts);
                return 0;
            case NGAPT_K_RBGS:
                if (prec)
                    launch_sweep<float>(s, L0.g, L0.s.c, L0.s.a0, L0.s.a1, L0.s.a2, h->r32, h->z32, L0.s.w, 0);
                else
                    launch_sweep<double>(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, h->r, h->z, L0.d.w, 0);
                return 0;
            case NGAPT_K_SWEEP2:
            case NGAPT_K_SWEEP2_ZERO: {
                const bool z = kid == NGAPT_K_SWEEP2_ZERO;
                if (prec)
                    launch_sweep2<float>(s, L0.g, L0.s.c, L0.s.a0, L0.s.a1, L0.s.a2, h->r32, z ? nullptr : h->z32,
                                         L0.s.w, 0);
                else
                    launch_sweep2<double>(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, h->r, z ? nullptr : h->z,
                                          L0.d.w, 0);
                return 0;
            }
            case NGAPT_K_RESTRICT: {
                if (h->nlev < 2) return NGAP_ERR_ARG;
                Level &C = h->lev[1];
                if (prec) {
                    launch_resid<float>(s, L0.g, L0.s.c, L0.s.a0, L0.s.a1, L0.s.a2, h->r32, h->z32, L0.s.w);
                    launch_gather<float>(s, L0.g, C.g, L0.cdir, L0.s.w, C.s.pm, C.s.pp, C.s.f);
                } else {
                    launch_resid<double>(s, L0.g, L0.d.c, L0.d.a0, L0.d.a1, L0.d.a2, h->r, h->z, L0.d.w);
                    launch_gather<double>(s, L0.g, C.g, L0.cdir, L0.d.w, C.d.pm, C.d.pp, C.d.f);
                }
                return 0;
            }
            case NGAPT_K_PROLONG: {
                if (h->nlev < 2) return NGAP_ERR_ARG;
                Level &C = h->lev[1];
                if (prec)
                    launch_prolong_to<float>(s, L0.g, C.g, L0.cdir, C.s.pm, C.s.pp, C.s.v, h->z32, h->z32);
                else
                    launch_prolong_to<double>(s, L0.g, C.g, L0.cdir, C.d.pm, C.d.pp, C.d.v, h->z, h->z);
                return 0;
            }
            case NGAPT_K_UPDATE: {
                int nb = grid_for(N);
                hipLaunchKernelGGL(k_update_xr<double>, dim3(nb), dim3(NT), 0, s, N, h->x, h->r,
                                   (const double *)h->p, (const double *)h->q, (const double *)h->scal,
                                   (float *)nullptr, h->parts);
                return 0;
            }
            case NGAPT_K_EXACT:
                return exact_residual(h, h->q, S_RRT);
            default:
                return NGAP_ERR_ARG;
        }
    };
    // byte model: every array touched once per launch
    double b;
    switch (kid) {
        case NGAPT_K_SPMV: b = 6.0 * w * N; break;
        case NGAPT_K_RBGS: b = 7.0 * w * N; break;  // full sweep: 4 coef + f + v in + v out
        case NGAPT_K_SWEEP2: b = 7.0 * w * N; break;  // two sweeps, the same arrays once
        case NGAPT_K_SWEEP2_ZERO: b = 6.0 * w * N; break;  // no v in
        case NGAPT_K_RESTRICT: b = (h->nlev > 1 ? (8.0 * w * N + 3.0 * w * h->lev[1].g.N) : 0.0); break;
        case NGAPT_K_PROLONG: b = (h->nlev > 1 ? (2.0 * w * N + 3.0 * w * h->lev[1].g.N) : 0.0); break;
        case NGAPT_K_UPDATE: b = 6.0 * 8.0 * N; break;
        case NGAPT_K_EXACT: b = (7.0 + 3.0) * 8.0 * N; break;
        default: return NGAP_ERR_ARG;
    }
    int rc = launch();  // warm-up
    if (rc) return rc;
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(e0, s));
    for (int r = 0; r < reps; r++) launch();
    HIPCHK(hipEventRecord(e1, s));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *avg_ms = ms / reps;
    *bytes = b;
    return 0;
}

}  // extern "C"
