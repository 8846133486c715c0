// fourier3d on the GPU: the FFT direct solve of a circulant stencil operator
// on a periodic uniform grid (fourier3d_class.f90:1103-1202): the circulance
// check, the placement of the stencil, the inversion of the transformed
// operator, the transforms with the spectral divide, the copy of the solution
// into sol and its ghost fill.
//
// The transforms are real-to-complex over the directions with more than one
// cell, x first. Where x is one of them and every length is a product of 2, 3,
// 5, 7, 11 and 13 of at most FFT_MAX, they are the kernels of this file: a
// solve is five passes over memory (x forward, y forward, z forward with the
// divide and z inverse, y inverse, x inverse into sol and its ghosts). 256^3:
// 346 us a solve, with the library 581; 90 x 75 x 64: 60 and 77 us. Against a
// solve in extended precision their error is about half of the library's
// (geometric mean over 90 grids of one to three directions).
//
// Elsewhere rocFFT (through hipFFT) transforms. The forward plan reads the
// interior of the caller's ghosted rhs in place (strided plan layout); the
// inverse one writes a dense array (rocFFT's two-dimensional complex-to-real
// plans with a strided output fail to execute), which one pass copies into the
// interior of sol. A solve is: forward transform, one pass over the half
// spectrum (zero mode, 1/F, normalisation), inverse transform, copy, ghost fill.
// The half spectrum (last transformed direction n/2+1 long) holds every mode
// of the reference's full complex transform, since F(-k) = conj F(k) for a
// real stencil and a real right-hand side.
#include <hip/hip_runtime.h>
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <type_traits>
#include <vector>

#include "ngapfft.h"

namespace {

constexpr int PT = 256;
constexpr int NB = 1024;  // blocks of the reductions (partials summed on the host)

struct Grid {
    int nx, ny, nz;          // interior
    int nxo, nyo, nzo;       // ghosted
    int gx, gy, gz;          // ghost widths
    int px, py, pz;          // periodic
    long long N, No;         // interior and ghosted cell counts
};

int blocks_for(long long n) {
    long long v = (n + PT - 1) / PT;
    if (v > 65535LL * 16) v = 65535LL * 16;
    return (int)(v < 1 ? 1 : v);
}

__device__ __forceinline__ long long ghosted(const Grid &g, int i, int j, int k) {
    return ((long long)(k + g.gz) * g.nyo + (j + g.gy)) * g.nxo + (i + g.gx);
}

// count the interior cells whose stencil differs from the first interior
// cell's by more than tol in any entry (fourier3d_class.f90:1118-1126)
__global__ void __launch_bounds__(PT) k_circulant(Grid g, int nst, const double *__restrict__ opr, double tol,
                                                  int *__restrict__ part) {
    __shared__ int sm[PT];
    const double *ref = opr + (size_t)nst * ghosted(g, 0, 0, 0);
    int bad = 0;
    for (long long q = blockIdx.x * (long long)PT + threadIdx.x; q < g.N; q += (long long)gridDim.x * PT) {
        const int i = (int)(q % g.nx);
        const long long r = q / g.nx;
        const int j = (int)(r % g.ny), k = (int)(r / g.ny);
        const double *o = opr + (size_t)nst * ghosted(g, i, j, k);
        for (int s = 0; s < nst; s++)
            if (fabs(o[s] - ref[s]) > tol) {
                bad = 1;
                break;
            }
    }
    sm[threadIdx.x] = bad;
    __syncthreads();
    for (int w = PT / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) sm[threadIdx.x] += sm[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sm[0];
}

__global__ void __launch_bounds__(PT) k_zero(double *__restrict__ a, long long n) {
    for (long long q = blockIdx.x * (long long)PT + threadIdx.x; q < n; q += (long long)gridDim.x * PT) a[q] = 0.0;
}

// the first interior cell's stencil at its offsets modulo the grid
// (fourier3d_class.f90:1128-1137), into the interior of a ghosted-layout
// array; one thread, in stencil order
__global__ void k_place(Grid g, int nst, const int *__restrict__ stc, const double *__restrict__ opr,
                        double *__restrict__ kern) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const double *ref = opr + (size_t)nst * ghosted(g, 0, 0, 0);
    for (int s = 0; s < nst; s++) {
        int i = stc[s] % g.nx, j = stc[s + nst] % g.ny, k = stc[s + 2 * nst] % g.nz;
        if (i < 0) i += g.nx;
        if (j < 0) j += g.ny;
        if (k < 0) k += g.nz;
        kern[ghosted(g, i, j, k)] += ref[s];
    }
}

// zero mode to 1, count |F| < 1000 eps, invert, count NaN
// (fourier3d_class.f90:1142-1160)
// (rows of `pitch` modes, `len` of them in use)
__global__ void __launch_bounds__(PT) k_invert(long long M, int pitch, int len, double2 *__restrict__ F,
                                               int *__restrict__ part_small, int *__restrict__ part_nan) {
    __shared__ int s0[PT], s1[PT];
    int small = 0, nan = 0;
    for (long long m = blockIdx.x * (long long)PT + threadIdx.x; m < M; m += (long long)gridDim.x * PT) {
        if (m % pitch >= len) continue;
        double2 f = F[m];
        if (m == 0) f = make_double2(1.0, 0.0);
        if (hypot(f.x, f.y) < 1000.0 * DBL_EPSILON) small++;
        const double d = f.x * f.x + f.y * f.y;
        const double2 r = make_double2(f.x / d, -f.y / d);
        if (isnan(hypot(r.x, r.y))) nan++;
        F[m] = r;
    }
    s0[threadIdx.x] = small;
    s1[threadIdx.x] = nan;
    __syncthreads();
    for (int w = PT / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            s0[threadIdx.x] += s0[threadIdx.x + w];
            s1[threadIdx.x] += s1[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part_small[blockIdx.x] = s0[0];
        part_nan[blockIdx.x] = s1[0];
    }
}

// G = G / F with the zero mode of G set to 0 (fourier3d_class.f90:1039-1040,
// 1186-1187) and the three 1/n of the inverse transforms folded in
__global__ void __launch_bounds__(PT) k_divide(long long M, double2 *__restrict__ G, const double2 *__restrict__ Finv,
                                               double scale) {
    for (long long m = blockIdx.x * (long long)PT + threadIdx.x; m < M; m += (long long)gridDim.x * PT) {
        const double2 a = m == 0 ? make_double2(0.0, 0.0) : G[m];
        const double2 b = Finv[m];
        G[m] = make_double2((a.x * b.x - a.y * b.y) * scale, (a.x * b.y + a.y * b.x) * scale);
    }
}

// interior of a ghosted array from a dense x-fastest one
__global__ void __launch_bounds__(PT) k_put(Grid g, const double *__restrict__ d, double *__restrict__ a) {
    for (long long q = blockIdx.x * (long long)PT + threadIdx.x; q < g.N; q += (long long)gridDim.x * PT) {
        const int i = (int)(q % g.nx);
        const long long r = q / g.nx;
        a[ghosted(g, i, (int)(r % g.ny), (int)(r / g.ny))] = d[q];
    }
}

// ghost fill of one direction, as cfg%sync does on one rank
// (pgrid_class.f90:459-516): the 2*w ghost layers of direction ax take the
// periodic image, over the whole ghosted extent of the other two directions
// (so the passes x, then y, then z also fill edges and corners). The cells
// read lie inside the box in direction ax and are not written by the pass.
__global__ void __launch_bounds__(PT) k_sync_dir(Grid g, int ax, double *a) {
    const int n = ax == 0 ? g.nx : (ax == 1 ? g.ny : g.nz);
    const int w = ax == 0 ? g.gx : (ax == 1 ? g.gy : g.gz);
    const int e0 = ax == 0 ? g.nyo : g.nxo;  // the other two ghosted extents
    const int e1 = ax == 2 ? g.nyo : g.nzo;
    const long long total = (long long)e0 * e1 * 2 * w;
    for (long long q = blockIdx.x * (long long)PT + threadIdx.x; q < total; q += (long long)gridDim.x * PT) {
        const int l = (int)(q % (2 * w));
        const long long r = q / (2 * w);
        const int u = (int)(r % e0), v = (int)(r / e0);
        // ghost layer l: ghosted index 0..w-1 (below) or n+w..n+2w-1 (above),
        // box coordinate l-w or n+l-w; its image is the box coordinate modulo n
        const int gidx = l < w ? l : n + l;
        const int src = w + ((l - w) % n + n) % n;
        long long dst_off, src_off;
        if (ax == 0) {
            dst_off = ((long long)v * g.nyo + u) * g.nxo + gidx;
            src_off = ((long long)v * g.nyo + u) * g.nxo + src;
        } else if (ax == 1) {
            dst_off = ((long long)v * g.nyo + gidx) * g.nxo + u;
            src_off = ((long long)v * g.nyo + src) * g.nxo + u;
        } else {
            dst_off = ((long long)gidx * g.nyo + v) * g.nxo + u;
            src_off = ((long long)src * g.nyo + v) * g.nxo + u;
        }
        a[dst_off] = a[src_off];
    }
}

// ------------------------------------------------------------------ transforms in LDS
// A transform of length n = r_0 r_1 ... (r of 2, 3, 4, 5, 7, 8, 11, 13; n <=
// FFT_MAX) decimated in frequency: pass p combines the r_p elements m_p =
// n / (r_0 .. r_p) apart and stores them where they were, so that a tile of
// lines is transformed in place in LDS with one barrier a pass; the first pass
// reads from memory and the last one writes to it. The modes end up in
// digit-reversed order and stay there: the operator's transform has the same
// order, the divide is pointwise, and the inverse runs the passes backwards.
constexpr int FFT_MAX = 1024;  // 8 lines of 16 bytes a cell: 128 KB of LDS
constexpr int FT = 256;                // threads of a row workgroup at most
constexpr int LB = 3, LINES = 1 << LB;  // lines of a column tile
struct FftDim {
    int n, np;
    int r[10], m[10];
    unsigned magic[10];  // 2^32 / m rounded up: g / m for g m < 2^32, m > 1
    const double2 *w;    // exp(-2 pi i k / n), k < n
    const unsigned short *pos;  // where mode k is
};

__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cmulc(double2 a, double2 b) {  // a conj(b)
    return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
template <bool INV>
__device__ __forceinline__ double2 mul_i(double2 a) {  // by -i (forward), i (inverse)
    return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

template <bool INV>
__device__ __forceinline__ void dft4(double2 &a, double2 &b, double2 &c, double2 &d) {
    const double2 s0 = cadd(a, c), d0 = csub(a, c), s1 = cadd(b, d), d1 = mul_i<INV>(csub(b, d));
    a = cadd(s0, s1);
    c = csub(s0, s1);
    b = cadd(d0, d1);
    d = csub(d0, d1);
}

// v_k = sum_q v_q w^(qk), w the R-th root of unity; w: the table of n, whose
// entries n/R apart are that root's powers
template <int R, bool INV>
__device__ __forceinline__ void dft(double2 (&v)[R], const double2 *w, int n) {
    if constexpr (R == 2) {
        const double2 t = csub(v[0], v[1]);
        v[0] = cadd(v[0], v[1]);
        v[1] = t;
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        constexpr double h = 0.70710678118654752440;  // sqrt(1/2)
        dft4<INV>(v[0], v[2], v[4], v[6]);
        dft4<INV>(v[1], v[3], v[5], v[7]);
        const double2 t = mul_i<INV>(v[3]), u = mul_i<INV>(v[7]);
        const double2 o1 = make_double2(h * (v[3].x + t.x), h * (v[3].y + t.y));
        const double2 o2 = mul_i<INV>(v[5]);
        const double2 o3 = make_double2(h * (u.x - v[7].x), h * (u.y - v[7].y));
        const double2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
        v[0] = cadd(e0, o0);
        v[4] = csub(e0, o0);
        v[1] = cadd(e1, o1);
        v[5] = csub(e1, o1);
        v[2] = cadd(e2, o2);
        v[6] = csub(e2, o2);
        v[3] = cadd(e3, o3);
        v[7] = csub(e3, o3);
    } else {
        // odd: sums and differences of the pairs q, R - q against cosines and sines
        constexpr int H = (R - 1) / 2;
        double2 s[H], d[H], c[H];
        const int step = n / R;
#pragma unroll
        for (int q = 0; q < H; q++) {
            s[q] = cadd(v[q + 1], v[R - 1 - q]);
            d[q] = csub(v[q + 1], v[R - 1 - q]);
            c[q] = w[(q + 1) * step];
        }
        double2 t = v[0];
#pragma unroll
        for (int q = 0; q < H; q++) t = cadd(t, s[q]);
        const double2 x0 = v[0];
        v[0] = t;
#pragma unroll
        for (int k = 1; k <= H; k++) {
            double2 e = x0, o = make_double2(0.0, 0.0);
#pragma unroll
            for (int q = 1; q <= H; q++) {
                const int x = q * k % R, z = x <= H ? x : R - x;  // a folded constant
                const double cs = c[z - 1].x, sn = x <= H ? c[z - 1].y : -c[z - 1].y;
                e.x += s[q - 1].x * cs;
                e.y += s[q - 1].y * cs;
                o.x += d[q - 1].x * sn;
                o.y += d[q - 1].y * sn;
            }
            // i o (forward; the table's sines are already negative), -i o (inverse)
            const double2 io = INV ? make_double2(o.y, -o.x) : make_double2(-o.y, o.x);
            v[k] = cadd(e, io);
            v[R - k] = csub(e, io);
        }
    }
}

// one butterfly's r elements: twiddles before the inverse, after the forward one
template <int R, bool INV>
__device__ __forceinline__ void butterfly(double2 (&v)[R], const double2 *w, int n, int j, int m) {
    const int lj = n / (R * m) * j;
    if (INV) {
#pragma unroll
        for (int q = 1; q < R; q++) v[q] = cmulc(v[q], w[lj * q]);
        dft<R, true>(v, w, n);
    } else {
        dft<R, false>(v, w, n);
#pragma unroll
        for (int q = 1; q < R; q++) v[q] = cmul(v[q], w[lj * q]);
    }
}

__device__ __forceinline__ int div_m(int g, int m, unsigned magic) { return m == 1 ? g : (int)__umulhi((unsigned)g, magic); }

// BIG: with the radices 7, 11 and 13, which take up to twice the registers
template <bool BIG, typename Run>
__device__ __forceinline__ void by_radix(int r, Run run) {
    if (r == 8) {
        run(std::integral_constant<int, 8>());
    } else if (r == 4) {
        run(std::integral_constant<int, 4>());
    } else if (r == 2) {
        run(std::integral_constant<int, 2>());
    } else if (r == 3) {
        run(std::integral_constant<int, 3>());
    } else if (!BIG || r == 5) {
        run(std::integral_constant<int, 5>());
    } else if constexpr (BIG) {
        if (r == 7)
            run(std::integral_constant<int, 7>());
        else if (r == 11)
            run(std::integral_constant<int, 11>());
        else
            run(std::integral_constant<int, 13>());
    }
}

// Lines across rows (y and z). A workgroup transforms 8 adjacent ones:
// whole 128-byte lines of every row, a row of the half spectrum being padded to
// 8 modes for that. FWD and INV in place; DIVIDE: forward, times finv, inverse,
// in one pass over memory, the last forward and the first inverse pass in
// registers. line l of outer o starts at o * ostride + l; its elements are es
// apart; lines whose x is padding are left out.
// Bound by memory: at 256^3 (129 x 256 x 256 modes, 270 MB in and out) 55 us a plain
// pass, the library's 82; the divide (405 MB) 103 us, two library passes and a
// divide 221.
enum { FWD, INV, DIVIDE };
// Threads: one per radix-8 butterfly of a pass, at most 256, or so many that the
// workgroups that fit a CU's LDS fill its 16 waves (8 of a BIG kernel's): lines of
// more than 568 cells leave one and with 256 threads its latency bare
// (1024^2 x 32: 1080 us a solve with 256 threads, 917 now; 16 x 1024 x 16: 105 and
// 79 us, the library 84 to 99). Other counts than powers of two leave SIMDs uneven
// (300^3 with 320 threads: 788 us against 685).
constexpr size_t CU_LDS = 160 * 1024;
template <int MODE, bool BIG>
__global__ void __launch_bounds__(BIG ? 512 : 1024) k_fft_col(FftDim D, const double2 *__restrict__ finv, double2 *a, int nlines,
                                                long long es, long long ostride, int pitch, int nxh,
                                                double scale) {
    extern __shared__ double2 sm[];
    const int n = D.n, T = blockDim.x;
    double2 *w = sm, *t = sm + n;
    for (int i = threadIdx.x; i < n; i += T) w[i] = D.w[i];
    const int c = threadIdx.x & (LINES - 1), g0 = threadIdx.x >> LB, gs = T >> LB;
    const int line = blockIdx.x * LINES + c;
    const bool on = line < nlines && line % pitch < nxh;
    const long long base = (long long)blockIdx.y * ostride + line;
    const bool zero = base == 0;  // the line of the zero mode
    double2 *__restrict__ p = a + base;
    const double2 *__restrict__ fi = MODE == DIVIDE ? finv + base : nullptr;
    __syncthreads();
    const int np = D.np;
    const int total = MODE == DIVIDE ? 2 * np - 1 : np;
    for (int k = 0; k < total; k++) {
        // the pass of this step and where its elements are
        const bool inv = MODE == INV || (MODE == DIVIDE && k >= np);
        const int ps = MODE == INV ? np - 1 - k : (MODE == DIVIDE && k >= np ? 2 * np - 2 - k : k);
        const bool in = k == 0, out = k == total - 1, mid = MODE == DIVIDE && k == np - 1;
        const int r = D.r[ps], m = D.m[ps];
        const unsigned magic = D.magic[ps];
        const int ng = n / r;
        auto run = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            if (!on) return;
            for (int g = g0; g < ng; g += gs) {
                const int l = div_m(g, m, magic), j = g - l * m, b = l * R * m + j;
                double2 v[R];
#pragma unroll
                for (int q = 0; q < R; q++) v[q] = in ? p[(b + q * m) * es] : t[((b + q * m) << LB) + c];
                if (mid) {
                    double2 f[R];
#pragma unroll
                    for (int q = 0; q < R; q++) f[q] = fi[(b + q * m) * es];
                    dft<R, false>(v, w, n);  // the last pass: m = 1, no twiddles
#pragma unroll
                    for (int q = 0; q < R; q++) {
                        v[q] = cmul(v[q], f[q]);
                        v[q].x *= scale;
                        v[q].y *= scale;
                    }
                    if (zero && b == 0) v[0] = make_double2(0.0, 0.0);
                    dft<R, true>(v, w, n);
                } else if (MODE != FWD && inv) {
                    butterfly<R, true>(v, w, n, j, m);
                } else {
                    butterfly<R, false>(v, w, n, j, m);
                }
#pragma unroll
                for (int q = 0; q < R; q++) {
                    if (out)
                        p[(b + q * m) * es] = v[q];
                    else
                        t[((b + q * m) << LB) + c] = v[q];
                }
            }
        };
        by_radix<BIG>(r, run);
        if (!out) __syncthreads();
    }
}

__device__ __forceinline__ int padx(int i) { return i + (i >> 3); }  // strides of 8 over all banks

// Rows, real to half spectrum (256^3, 269 MB: 61 us, the library's 56): two rows as the real and the imaginary part of one
// complex row, separated afterwards. src: the first interior cell of a ghosted
// array; row q is row (q % ny, q / ny). pairs rows pairs per workgroup.
template <bool BIG>
__global__ void __launch_bounds__(FT) k_fft_x(FftDim D, Grid G, const double *__restrict__ src, double2 *__restrict__ dst,
                                              int nrows, int pairs, int pitch) {
    extern __shared__ double2 sm[];
    const int n = D.n, ld = padx(n) + 1, nxh = n / 2 + 1, T = blockDim.x;
    double2 *w = sm, *t = sm + n;
    unsigned short *pos = reinterpret_cast<unsigned short *>(t + pairs * ld);
    for (int i = threadIdx.x; i < n; i += T) {
        w[i] = D.w[i];
        pos[i] = D.pos[i];
    }
    const int row0 = blockIdx.x * pairs * 2, my = min(pairs, (nrows - row0 + 1) / 2);
    __syncthreads();
    for (int k = 0; k < D.np; k++) {
        const int r = D.r[k], m = D.m[k], ng = n / r;
        const unsigned magic = D.magic[k];
        auto run = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            for (int e = threadIdx.x; e < ng * my; e += T) {
                const int pr = e / ng, g = e - pr * ng;
                const int l = div_m(g, m, magic), j = g - l * m, b = l * R * m + j;
                double2 *__restrict__ tl = t + pr * ld;
                double2 v[R];
                if (k == 0) {
                    const int qa = row0 + 2 * pr, qb = qa + 1;
                    const double *__restrict__ ra = src + ((long long)(qa / G.ny) * G.nyo + qa % G.ny) * G.nxo;
                    const double *__restrict__ rb = src + ((long long)(qb / G.ny) * G.nyo + qb % G.ny) * G.nxo;
                    const bool two = qb < nrows;
#pragma unroll
                    for (int q = 0; q < R; q++) v[q] = make_double2(ra[b + q * m], two ? rb[b + q * m] : 0.0);
                } else {
#pragma unroll
                    for (int q = 0; q < R; q++) v[q] = tl[padx(b + q * m)];
                }
                butterfly<R, false>(v, w, n, j, m);
#pragma unroll
                for (int q = 0; q < R; q++) tl[padx(b + q * m)] = v[q];
            }
        };
        by_radix<BIG>(r, run);
        __syncthreads();
    }
    for (int e = threadIdx.x; e < nxh * my; e += T) {
        const int pr = e / nxh, k = e - pr * nxh;
        const double2 *__restrict__ tl = t + pr * ld;
        const double2 a = tl[padx(pos[k])], b = tl[padx(pos[k == 0 ? 0 : n - k])];
        const long long q = row0 + 2 * pr;
        dst[q * pitch + k] = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
        if (q + 1 < nrows) dst[(q + 1) * pitch + k] = make_double2(0.5 * (a.y + b.y), 0.5 * (b.x - a.x));
    }
}

// Half spectrum to real rows, the inverse of k_fft_x, into the interior of a
// ghosted array and, with `images`, into every ghost cell that is a periodic
// image of it (each ghost width at most the box's length): 256^3: 69 us; the
// library's transform, a copy into the box and the three ghost passes took
// 49 + 53 + 16.
template <bool BIG>
__global__ void __launch_bounds__(FT) k_fft_xinv(FftDim D, Grid G, const double2 *__restrict__ src, double *__restrict__ dst,
                                                 int nrows, int pairs, int pitch, int images) {
    extern __shared__ double2 sm[];
    const int n = D.n, ld = padx(n) + 1, nxh = n / 2 + 1, T = blockDim.x;
    double2 *w = sm, *t = sm + n;
    unsigned short *pos = reinterpret_cast<unsigned short *>(t + pairs * ld);
    for (int i = threadIdx.x; i < n; i += T) {
        w[i] = D.w[i];
        pos[i] = D.pos[i];
    }
    const int row0 = blockIdx.x * pairs * 2, my = min(pairs, (nrows - row0 + 1) / 2);
    __syncthreads();
    for (int e = threadIdx.x; e < nxh * my; e += T) {
        const int pr = e / nxh, k = e - pr * nxh;
        double2 *__restrict__ tl = t + pr * ld;
        const long long q = row0 + 2 * pr;
        double2 a = src[q * pitch + k], b = q + 1 < nrows ? src[(q + 1) * pitch + k] : make_double2(0.0, 0.0);
        // the modes that are their own conjugates are real
        if (k == 0 || 2 * k == n) a.y = b.y = 0.0;
        tl[padx(pos[k])] = make_double2(a.x - b.y, a.y + b.x);
        if (k > 0 && 2 * k != n) tl[padx(pos[n - k])] = make_double2(a.x + b.y, b.x - a.y);
    }
    __syncthreads();
    const long long splane = (long long)G.nxo * G.nyo;
    for (int k = D.np - 1; k >= 0; k--) {
        const int r = D.r[k], m = D.m[k], ng = n / r;
        const unsigned magic = D.magic[k];
        auto run = [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            for (int e = threadIdx.x; e < ng * my; e += T) {
                const int pr = e / ng, g = e - pr * ng;
                const int l = div_m(g, m, magic), j = g - l * m, b = l * R * m + j;
                double2 *__restrict__ tl = t + pr * ld;
                double2 v[R];
#pragma unroll
                for (int q = 0; q < R; q++) v[q] = tl[padx(b + q * m)];
                butterfly<R, true>(v, w, n, j, m);
                if (k > 0) {
#pragma unroll
                    for (int q = 0; q < R; q++) tl[padx(b + q * m)] = v[q];
                    continue;
                }
                for (int h = 0; h < 2; h++) {
                    const int qr = row0 + 2 * pr + h;
                    if (qr >= nrows) break;
                    const int jy = qr % G.ny, kz = qr / G.ny;
                    for (int iz = -1; iz <= 1; iz++) {
                        const int zz = kz + iz * G.nz + G.gz;
                        if (iz != 0 && (!images || zz < 0 || zz >= G.nzo)) continue;
                        for (int iy = -1; iy <= 1; iy++) {
                            const int yy = jy + iy * G.ny + G.gy;
                            if (iy != 0 && (!images || yy < 0 || yy >= G.nyo)) continue;
                            double *__restrict__ o = dst + zz * splane + (long long)yy * G.nxo + G.gx;
#pragma unroll
                            for (int q = 0; q < R; q++) {
                                const int x = b + q * m;
                                const double val = h == 0 ? v[q].x : v[q].y;
                                o[x] = val;
                                if (images && x < G.gx) o[x + n] = val;
                                if (images && x >= n - G.gx) o[x - n] = val;
                            }
                        }
                    }
                }
            }
        };
        by_radix<BIG>(r, run);
        __syncthreads();
    }
}

int sync_all(hipStream_t s, const Grid &g, double *a) {
    const int per[3] = {g.px, g.py, g.pz}, w[3] = {g.gx, g.gy, g.gz};
    const long long e[3] = {(long long)g.nyo * g.nzo, (long long)g.nxo * g.nzo, (long long)g.nxo * g.nyo};
    for (int ax = 0; ax < 3; ax++) {
        if (!per[ax] || w[ax] == 0) continue;
        hipLaunchKernelGGL(k_sync_dir, dim3(blocks_for(e[ax] * 2 * w[ax])), dim3(PT), 0, s, g, ax, a);
    }
    return 0;
}

}  // namespace

struct ngap_fft {
    Grid g{};
    int nst = 0;
    int device = 0;
    int rank = 0;       // directions with more than one cell
    long long M = 1;    // complex modes of the half spectrum (with padding)
    int pitch = 1, nxh = 1;    // modes of a row, allocated and in use
    bool own = false;          // the transforms of this file, else the library's
    bool images = false;       // the inverse fills the ghosts
    FftDim D[3]{};             // x, y, z
    hipStream_t s = nullptr;
    hipfftHandle fwd = 0, inv = 0;
    bool have_fwd = false, have_inv = false, setup_done = false;
    int *d_stc = nullptr, *d_part = nullptr;
    double *d_kern = nullptr;  // scratch: the stencil in ghosted layout (setup), the dense solution (solve)
    long long off = 0;         // offset of the first interior cell in a ghosted array
    double2 *d_spec = nullptr, *d_finv = nullptr;
    double *d_io = nullptr;  // ghosted staging for the host entry points
    hipEvent_t e0 = nullptr, e1 = nullptr;
    double last_ms = 0.0;
    std::vector<void *> allocs;
    ~ngap_fft() {
        if (have_fwd) (void)hipfftDestroy(fwd);
        if (have_inv) (void)hipfftDestroy(inv);
        for (void *q : allocs) (void)hipFree(q);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        if (s) (void)hipStreamDestroy(s);
    }
};

namespace {

template <typename T>
int dalloc(ngap_fft *F, T **p, size_t n) {
    void *q = nullptr;
    if (hipMalloc(&q, sizeof(T) * (n ? n : 1)) != hipSuccess) return NGAP_ERR_ALLOC;
    F->allocs.push_back(q);
    *p = (T *)q;
    return 0;
}

// a failed runtime or transform call: name it on stderr, return NGAP_ERR_HIP
int fail(const char *where, int code) {
    std::fprintf(stderr, "[ngap_fft] %s failed (%d)\n", where, code);
    return NGAP_ERR_HIP;
}

int fin(ngap_fft *F) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(hipGetErrorString(e), (int)e);
    e = hipStreamSynchronize(F->s);
    return e == hipSuccess ? 0 : fail(hipGetErrorString(e), (int)e);
}

int sum_parts(ngap_fft *F, const int *d, long long *out) {
    std::vector<int> h(NB);
    if (hipMemcpy(h.data(), d, sizeof(int) * NB, hipMemcpyDeviceToHost) != hipSuccess) return NGAP_ERR_HIP;
    long long t = 0;
    for (int v : h) t += v;
    *out = t;
    return 0;
}

// r_p and m_p of n; false if n has other factors or is too long
bool factor(int n, FftDim *D) {
    if (n < 2 || n > FFT_MAX) return false;
    static const int radix[] = {13, 11, 7, 5, 3};
    D->n = n;
    D->np = 0;
    int rest = n;
    while (rest % 8 == 0) D->r[D->np++] = 8, rest /= 8;
    if (rest % 4 == 0) D->r[D->np++] = 4, rest /= 4;
    if (rest % 2 == 0) D->r[D->np++] = 2, rest /= 2;
    for (int r : radix)
        while (rest % r == 0) D->r[D->np++] = r, rest /= r;
    if (rest != 1) return false;
    int m = n;
    for (int p = 0; p < D->np; p++) {
        m /= D->r[p];
        D->m[p] = m;
        D->magic[p] = m > 1 ? (unsigned)(((1ULL << 32) + m - 1) / m) : 0;
    }
    return true;
}

// tables of one direction
int plan_dim(ngap_fft *F, FftDim *D) {
    const int n = D->n;
    std::vector<double2> w(n);
    std::vector<unsigned short> pos(n);
    const long double tau = 2.0L * acosl(-1.0L);
    for (int k = 0; k < n; k++) {
        w[k] = make_double2((double)cosl(tau * k / n), (double)-sinl(tau * k / n));
        int f = k, at = 0;
        for (int p = 0; p < D->np; p++) {
            at += f % D->r[p] * D->m[p];
            f /= D->r[p];
        }
        pos[k] = (unsigned short)at;
    }
    double2 *dw = nullptr;
    unsigned short *dp = nullptr;
    int rc = dalloc(F, &dw, n);
    if (!rc) rc = dalloc(F, &dp, n);
    if (!rc && (hipMemcpy(dw, w.data(), sizeof(double2) * n, hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(dp, pos.data(), sizeof(unsigned short) * n, hipMemcpyHostToDevice) != hipSuccess))
        rc = NGAP_ERR_HIP;
    D->w = dw;
    D->pos = dp;
    return rc;
}

// Row pairs of a workgroup: about 2048 cells, so that 256 threads have one
// radix-8 butterfly each, but fewer where that leaves less than two workgroups
// per CU.
int row_pairs(const Grid &g) {
    int pr = std::min(16, std::max(1, 2048 / g.nx));
    while (pr > 1 && (long long)g.ny * g.nz / (2 * pr) < 512) pr /= 2;
    return pr;
}
int threads_for(int cells, int most = FT) { return std::min(most, std::max(64, (cells / 8 + 63) / 64 * 64)); }
size_t row_lds(int n, int pr) { return sizeof(double2) * (n + (size_t)pr * (n + n / 8 + 1)) + sizeof(short) * n; }
size_t col_lds(int n) { return sizeof(double2) * (n + (size_t)n * LINES); }

bool big(const FftDim &D) {
    for (int p = 0; p < D.np; p++)
        if (D.r[p] == 7 || D.r[p] > 8) return true;
    return false;
}

int col_threads(const FftDim &D) {
    const size_t fit = CU_LDS / col_lds(D.n);
    const int most = big(D) ? (fit > 1 ? 256 : 512) : (fit > 2 ? 256 : (fit > 1 ? 512 : 1024));
    return threads_for(D.n * LINES, most);
}

void rows_fwd(ngap_fft *F, const double *src, double2 *dst) {
    const int rows = F->g.ny * F->g.nz, pr = row_pairs(F->g);
    hipLaunchKernelGGL(big(F->D[0]) ? k_fft_x<true> : k_fft_x<false>, dim3((unsigned)((rows + 2 * pr - 1) / (2 * pr))),
                       dim3(threads_for(pr * F->g.nx)), row_lds(F->g.nx, pr), F->s, F->D[0], F->g, src, dst, rows, pr, F->pitch);
}

void rows_inv(ngap_fft *F, const double2 *src, double *dst) {
    const int rows = F->g.ny * F->g.nz, pr = row_pairs(F->g);
    hipLaunchKernelGGL(big(F->D[0]) ? k_fft_xinv<true> : k_fft_xinv<false>,
                       dim3((unsigned)((rows + 2 * pr - 1) / (2 * pr))), dim3(threads_for(pr * F->g.nx)), row_lds(F->g.nx, pr), F->s, F->D[0], F->g,
                       src, dst, rows, pr, F->pitch, F->images ? 1 : 0);
}

template <int MODE>
auto col_kernel(const FftDim &D) {
    return big(D) ? k_fft_col<MODE, true> : k_fft_col<MODE, false>;
}

template <int MODE>
void cols(ngap_fft *F, int ax, double2 *a, double scale) {
    const Grid &g = F->g;
    const int n = F->D[ax].n;
    const long long row = F->pitch, plane = row * g.ny;
    const int lines = (int)(ax == 1 ? row : plane);
    hipLaunchKernelGGL(col_kernel<MODE>(F->D[ax]), dim3((unsigned)((lines + LINES - 1) / LINES), ax == 1 ? g.nz : 1),
                       dim3(col_threads(F->D[ax])), col_lds(n), F->s, F->D[ax], (const double2 *)F->d_finv, a, lines,
                       ax == 1 ? row : plane, plane, F->pitch, F->nxh, scale);
}

// More than 64 KB of LDS is asked for by name. The limit belongs to the kernel, not
// to a handle: always the largest tile's, so that no handle lowers another's.
bool allow_lds(const FftDim &D) {
    if (col_lds(D.n) <= 65536) return true;
    const void *k[] = {(const void *)col_kernel<FWD>(D), (const void *)col_kernel<INV>(D),
                       (const void *)col_kernel<DIVIDE>(D)};
    for (const void *q : k)
        if (hipFuncSetAttribute(q, hipFuncAttributeMaxDynamicSharedMemorySize, (int)col_lds(FFT_MAX)) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
    return true;
}

// own transforms: the operator's spectrum, and a whole solve
void own_forward(ngap_fft *F, const double *src, double2 *dst) {
    rows_fwd(F, src, dst);
    if (F->g.ny > 1) cols<FWD>(F, 1, dst, 1.0);
    if (F->g.nz > 1) cols<FWD>(F, 2, dst, 1.0);
}

void own_solve(ngap_fft *F, const double *src, double *dst) {
    const Grid &g = F->g;
    const double scale = 1.0 / ((double)g.nx * g.ny * g.nz);
    rows_fwd(F, src, F->d_spec);
    if (g.nz > 1) {
        if (g.ny > 1) cols<FWD>(F, 1, F->d_spec, 1.0);
        cols<DIVIDE>(F, 2, F->d_spec, scale);
        if (g.ny > 1) cols<INV>(F, 1, F->d_spec, 1.0);
    } else if (g.ny > 1) {
        cols<DIVIDE>(F, 1, F->d_spec, scale);
    } else {
        hipLaunchKernelGGL(k_divide, dim3(blocks_for(F->M)), dim3(PT), 0, F->s, F->M, F->d_spec,
                           (const double2 *)F->d_finv, scale);
    }
    rows_inv(F, F->d_spec, dst);
}

int setup_from(ngap_fft *F, const double *d_opr, double tol) {
    const Grid &g = F->g;
    F->setup_done = false;
    hipLaunchKernelGGL(k_circulant, dim3(NB), dim3(PT), 0, F->s, g, F->nst, d_opr, tol, F->d_part);
    int rc = fin(F);
    long long bad = 0;
    if (!rc) rc = sum_parts(F, F->d_part, &bad);
    if (rc) return rc;
    if (bad) return NGAP_ERR_NOT_CIRCULANT;
    hipLaunchKernelGGL(k_zero, dim3(blocks_for(g.No)), dim3(PT), 0, F->s, F->d_kern, g.No);
    hipLaunchKernelGGL(k_place, dim3(1), dim3(64), 0, F->s, g, F->nst, (const int *)F->d_stc, d_opr, F->d_kern);
    if (F->own) {
        own_forward(F, F->d_kern + F->off, F->d_finv);
    } else if (F->rank > 0) {
        const hipfftResult r = hipfftExecD2Z(F->fwd, F->d_kern + F->off, (hipfftDoubleComplex *)F->d_finv);
        if (r != HIPFFT_SUCCESS) return fail("hipfftExecD2Z (setup)", (int)r);
    } else if (hipMemcpyAsync(F->d_finv, F->d_kern + F->off, sizeof(double), hipMemcpyDeviceToDevice, F->s) !=
               hipSuccess) {
        return NGAP_ERR_HIP;  // one cell: the transform is the value itself (imaginary part set below)
    }
    if (F->rank == 0) hipLaunchKernelGGL(k_zero, dim3(1), dim3(PT), 0, F->s, (double *)F->d_finv + 1, 1LL);
    hipLaunchKernelGGL(k_invert, dim3(NB), dim3(PT), 0, F->s, F->M, F->pitch, F->nxh, F->d_finv, F->d_part,
                       F->d_part + NB);
    rc = fin(F);
    long long small = 0, nan = 0;
    if (!rc) rc = sum_parts(F, F->d_part, &small);
    if (!rc) rc = sum_parts(F, F->d_part + NB, &nan);
    if (rc) return rc;
    if (small || nan) return NGAP_ERR_SINGULAR;
    F->setup_done = true;
    return 0;
}

int solve_on(ngap_fft *F, const double *d_rhs, double *d_sol) {
    const Grid &g = F->g;
    if (hipEventRecord(F->e0, F->s) != hipSuccess) return fail("hipEventRecord", 0);
    if (F->own) {
        own_solve(F, d_rhs + F->off, d_sol);
    } else if (F->rank > 0) {
        // the plans read the interior of rhs and write the interior of sol in place
        hipfftResult r = hipfftExecD2Z(F->fwd, const_cast<double *>(d_rhs) + F->off, (hipfftDoubleComplex *)F->d_spec);
        if (r != HIPFFT_SUCCESS) return fail("hipfftExecD2Z", (int)r);
        hipLaunchKernelGGL(k_divide, dim3(blocks_for(F->M)), dim3(PT), 0, F->s, F->M, F->d_spec,
                           (const double2 *)F->d_finv, 1.0 / ((double)g.nx * g.ny * g.nz));
        r = hipfftExecZ2D(F->inv, (hipfftDoubleComplex *)F->d_spec, F->d_kern);
        if (r != HIPFFT_SUCCESS) return fail("hipfftExecZ2D", (int)r);
        hipLaunchKernelGGL(k_put, dim3(blocks_for(g.N)), dim3(PT), 0, F->s, g, (const double *)F->d_kern, d_sol);
    } else {
        hipLaunchKernelGGL(k_zero, dim3(1), dim3(PT), 0, F->s, d_sol + F->off, 1LL);  // the only mode is the zero mode
    }
    if (!F->images) sync_all(F->s, g, d_sol);
    if (hipEventRecord(F->e1, F->s) != hipSuccess) return fail("hipEventRecord", 0);
    int rc = fin(F);
    if (rc) return rc;
    float ms = 0.0f;
    const hipError_t e = hipEventElapsedTime(&ms, F->e0, F->e1);
    if (e != hipSuccess) return fail("hipEventElapsedTime", (int)e);
    F->last_ms = ms;
    return 0;
}

}  // namespace

extern "C" {

int ngap_fft_create(ngap_fft **fp, const ngap_grid *gr, int nst, const int *stc) {
    if (!fp) return NGAP_ERR_ARG;
    *fp = nullptr;
    if (!gr || !stc || nst < 1) return NGAP_ERR_ARG;
    Grid g{};
    g.nx = gr->imax_ - gr->imin_ + 1;
    g.ny = gr->jmax_ - gr->jmin_ + 1;
    g.nz = gr->kmax_ - gr->kmin_ + 1;
    g.nxo = gr->imaxo_ - gr->imino_ + 1;
    g.nyo = gr->jmaxo_ - gr->jmino_ + 1;
    g.nzo = gr->kmaxo_ - gr->kmino_ + 1;
    g.gx = gr->imin_ - gr->imino_;
    g.gy = gr->jmin_ - gr->jmino_;
    g.gz = gr->kmin_ - gr->kmino_;
    g.px = gr->xper;
    g.py = gr->yper;
    g.pz = gr->zper;
    if (g.nx < 1 || g.ny < 1 || g.nz < 1 || g.gx < 0 || g.gy < 0 || g.gz < 0) return NGAP_ERR_ARG;
    if (g.nx != gr->nx || g.ny != gr->ny || g.nz != gr->nz) return NGAP_ERR_ARG;  // one GPU holds the whole grid
    if (g.nxo != g.nx + 2 * g.gx || g.nyo != g.ny + 2 * g.gy || g.nzo != g.nz + 2 * g.gz) return NGAP_ERR_ARG;
    // fourier3d_class.f90:146-148: periodic wherever there is more than one cell
    if ((g.nx > 1 && !g.px) || (g.ny > 1 && !g.py) || (g.nz > 1 && !g.pz)) return NGAP_ERR_UNSUPPORTED;
    g.N = (long long)g.nx * g.ny * g.nz;
    g.No = (long long)g.nxo * g.nyo * g.nzo;
    if (nst * g.No >= (1LL << 40)) return NGAP_ERR_ARG;
    if (g.No >= (1LL << 31)) return NGAP_ERR_UNSUPPORTED;  // the plans' strides and distances are int
    ngap_fft *F = new ngap_fft();
    F->g = g;
    F->nst = nst;
    // transformed directions, slowest first, with their strides in the ghosted layout
    int dims[3], r = 0;
    long long str[3];
    if (g.nz > 1) dims[r] = g.nz, str[r++] = (long long)g.nxo * g.nyo;
    if (g.ny > 1) dims[r] = g.ny, str[r++] = g.nxo;
    if (g.nx > 1) dims[r] = g.nx, str[r++] = 1;
    F->rank = r;
    F->off = ((long long)g.gz * g.nyo + g.gy) * g.nxo + g.gx;
    F->M = 1;
    for (int d = 0; d + 1 < r; d++) F->M *= dims[d];
    if (r > 0) F->M *= dims[r - 1] / 2 + 1;
    F->own = g.nx > 1 && factor(g.nx, &F->D[0]) && (g.ny == 1 || factor(g.ny, &F->D[1])) &&
             (g.nz == 1 || factor(g.nz, &F->D[2])) && (long long)g.ny * g.nz < (1LL << 30) && g.nz < 65536 &&
             (g.ny == 1 || allow_lds(F->D[1])) && (g.nz == 1 || allow_lds(F->D[2]));  // else the library
    if (F->own) {
        F->nxh = g.nx / 2 + 1;
        F->pitch = (F->nxh + 7) / 8 * 8;
        F->M = (long long)F->pitch * g.ny * g.nz;
        F->images = g.px && g.py && g.pz && g.gx <= g.nx && g.gy <= g.ny && g.gz <= g.nz;
    } else {
        F->pitch = F->nxh = r > 0 ? dims[r - 1] / 2 + 1 : 1;
    }
    // real side: the ghosted array (embed[d] = stride ratio of consecutive
    // directions, the fastest stride as the element stride); complex side: the
    // dense half spectrum
    int rembed[3], cembed[3], dembed[3], rstride = r > 0 ? (int)str[r - 1] : 1;
    for (int d = 0; d < r; d++) {
        rembed[d] = d == 0 ? dims[0] : (int)(str[d - 1] / str[d]);
        cembed[d] = d == r - 1 ? dims[d] / 2 + 1 : dims[d];
        dembed[d] = dims[d];
    }
    int rc = hipGetDevice(&F->device) == hipSuccess ? 0 : NGAP_ERR_HIP;
    if (!rc) rc = hipStreamCreateWithFlags(&F->s, hipStreamNonBlocking) == hipSuccess ? 0 : NGAP_ERR_HIP;
    if (!rc) rc = hipEventCreate(&F->e0) == hipSuccess && hipEventCreate(&F->e1) == hipSuccess ? 0 : NGAP_ERR_HIP;
    if (!rc) rc = dalloc(F, &F->d_stc, 3 * (size_t)nst);
    if (!rc) rc = dalloc(F, &F->d_part, 2 * (size_t)NB);
    if (!rc) rc = dalloc(F, &F->d_kern, (size_t)g.No);
    if (!rc) rc = dalloc(F, &F->d_spec, (size_t)F->M);
    if (!rc) rc = dalloc(F, &F->d_finv, (size_t)F->M);
    if (!rc && hipMemcpy(F->d_stc, stc, sizeof(int) * 3 * nst, hipMemcpyHostToDevice) != hipSuccess) rc = NGAP_ERR_HIP;
    for (int d = 0; d < 3 && !rc && F->own; d++)
        if (F->D[d].n) rc = plan_dim(F, &F->D[d]);
    if (!rc && r > 0 && !F->own) {
        if (hipfftPlanMany(&F->fwd, r, dims, rembed, rstride, (int)g.No, cembed, 1, (int)F->M, HIPFFT_D2Z, 1) !=
            HIPFFT_SUCCESS)
            rc = NGAP_ERR_HIP;
        else
            F->have_fwd = true;
        if (!rc && hipfftPlanMany(&F->inv, r, dims, cembed, 1, (int)F->M, dembed, 1, (int)g.N, HIPFFT_Z2D, 1) !=
                       HIPFFT_SUCCESS)
            rc = NGAP_ERR_HIP;
        else if (!rc)
            F->have_inv = true;
        if (!rc && (hipfftSetStream(F->fwd, F->s) != HIPFFT_SUCCESS || hipfftSetStream(F->inv, F->s) != HIPFFT_SUCCESS))
            rc = NGAP_ERR_HIP;
    }
    if (rc) {
        delete F;
        return rc;
    }
    *fp = F;
    return 0;
}

int ngap_fft_setup_device(ngap_fft *f, const double *d_opr, double circ_tol) {
    if (!f || !d_opr || !(circ_tol >= 0.0)) return NGAP_ERR_ARG;
    if (hipSetDevice(f->device) != hipSuccess || hipDeviceSynchronize() != hipSuccess) return NGAP_ERR_HIP;
    return setup_from(f, d_opr, circ_tol);
}

int ngap_fft_setup(ngap_fft *f, const double *opr, double circ_tol) {
    if (!f || !opr || !(circ_tol >= 0.0)) return NGAP_ERR_ARG;
    if (hipSetDevice(f->device) != hipSuccess) return NGAP_ERR_HIP;
    const size_t n = (size_t)f->nst * f->g.No;
    double *d = nullptr;
    if (hipMalloc(&d, sizeof(double) * n) != hipSuccess) return NGAP_ERR_ALLOC;
    int rc = hipMemcpy(d, opr, sizeof(double) * n, hipMemcpyHostToDevice) == hipSuccess ? 0 : NGAP_ERR_HIP;
    if (!rc) rc = setup_from(f, d, circ_tol);
    (void)hipFree(d);
    return rc;
}

int ngap_fft_solve_device(ngap_fft *f, const double *d_rhs, double *d_sol) {
    if (!f || !d_rhs || !d_sol) return NGAP_ERR_ARG;
    if (!f->setup_done) return NGAP_ERR_NOT_SETUP;  // fourier3d_class.f90:1177
    if (hipSetDevice(f->device) != hipSuccess || hipDeviceSynchronize() != hipSuccess) return NGAP_ERR_HIP;
    return solve_on(f, d_rhs, d_sol);
}

int ngap_fft_solve(ngap_fft *f, const double *rhs, double *sol) {
    if (!f || !rhs || !sol) return NGAP_ERR_ARG;
    if (!f->setup_done) return NGAP_ERR_NOT_SETUP;
    if (hipSetDevice(f->device) != hipSuccess) return NGAP_ERR_HIP;
    const size_t n = (size_t)f->g.No;
    if (!f->d_io) {
        int rc = dalloc(f, &f->d_io, 2 * n);
        if (rc) return rc;
    }
    double *dr = f->d_io, *ds = f->d_io + n;
    // sol goes up too: ghosts of a non-periodic (one-cell) direction keep the caller's values
    if (hipMemcpy(dr, rhs, sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(ds, sol, sizeof(double) * n, hipMemcpyHostToDevice) != hipSuccess)
        return fail("hipMemcpy (upload)", 0);
    int rc = solve_on(f, dr, ds);
    if (!rc && hipMemcpy(sol, ds, sizeof(double) * n, hipMemcpyDeviceToHost) != hipSuccess)
        rc = fail("hipMemcpy (download)", 0);
    return rc;
}

int ngap_fft_destroy(ngap_fft *f) {
    if (!f) return NGAP_ERR_ARG;
    if (f->s) (void)hipStreamSynchronize(f->s);
    delete f;
    return 0;
}

int ngap_fft_last_ms(const ngap_fft *f, double *ms) {
    if (!f || !ms) return NGAP_ERR_ARG;
    *ms = f->last_ms;
    return 0;
}

}  // extern "C"
