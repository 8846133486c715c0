// Tiled level kernels (gfx950): SpMV, fused red/black Gauss-Seidel sweep,
// residual + restriction, prolongation + correction.
//
// Geometry: a level is n0 x n1 x n2 cells, p = i + n0*(j + n1*k) (int32 is
// enough for every level this solver allocates: N < 2^31 is checked at setup).
// Blocks tile the x-y plane; the SpMV and the sweep march through a chunk of
// z planes so each array element is read once and z neighbours come from
// registers.
#include <type_traits>

#include "ngap_internal.h"

namespace ngap {

namespace {

// coordinate wrapped into [0,n) for periodic directions; -1 outside a
// non-periodic box
__device__ __forceinline__ int wrapc(int i, int n, int per) {
    if (i >= 0 && i < n) return i;
    if (!per) return -1;
    i %= n;
    return i < 0 ? i + n : i;
}

// XCD-aware tile order. The dispatcher deals workgroups round-robin to the 8
// XCDs (workgroup b runs on XCD b % 8), each with its own L2. Remap the
// linear workgroup id so every XCD walks one contiguous range of tiles: tiles
// adjacent in y and z then share an L2, and their halo rows are hits.
// Bijective on [0, nb) for any nb.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    const int q = nb >> 3, r = nb & 7;
    const int x = b & 7, m = b >> 3;
    return x < r ? x * (q + 1) + m : r * (q + 1) + (x - r) * q + m;
}

// tile coordinates of this workgroup for a 1-D launch of gx*gy*gz groups
__device__ __forceinline__ void tile_of(int gx, int gy, int &bx, int &by, int &bz) {
    const int nb = gridDim.x;
    const int t = xcd_tile(blockIdx.x, nb);
    bx = t % gx;
    const int r = t / gx;
    by = r % gy;
    bz = r / gy;
}

}  // namespace

// ------------------------------------------------------------------ SpMV
// y = A x with the plane march; part (optional) gets one FP64 partial of
// <x, y> per block. Block (TX, TY) tiles x-y; blockIdx.z selects a z chunk.
// TX: the type x is stored in (FP32 search directions of the mixed solve
// with the FP64 operator); the product is formed in T.
template <typename T, typename TX = T>
__global__ void __launch_bounds__(256) k_apply_t(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                 const T *__restrict__ a1, const T *__restrict__ a2,
                                                 const TX *__restrict__ x, T *__restrict__ y,
                                                 double *__restrict__ part, int kc, int gx, int gy) {
    __shared__ double sm[4];
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int i = bx * blockDim.x + threadIdx.x;
    const int j = by * blockDim.y + threadIdx.y;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    double acc = 0.0;
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);
    if (i < n0 && j < n1 && k0 < k1) {
        const int im = nbm(i, n0, g.p0), ip = nbp(i, n0, g.p0);
        const int jm = nbm(j, n1, g.p1), jp = nbp(j, n1, g.p1);
        const int row = j * n0;
        const int om = im - i, op = ip - i;            // x offsets
        const int ym = (jm - j) * n0, yp = (jp - j) * n0;  // y offsets
        int km = nbm(k0, n2, g.p2);
        const int col = row + i;
        T xm = km >= 0 ? T(x[km * plane + col]) : T(0);
        T xc = T(x[k0 * plane + col]);
        T a2c = a2[k0 * plane + col];
        for (int k = k0; k < k1; k++) {
            const int p = k * plane + col;
            const int kp = nbp(k, n2, g.p2);
            const T xp = kp >= 0 ? T(x[kp * plane + col]) : T(0);
            const T a2p = kp >= 0 ? a2[kp * plane + col] : T(0);
            T s = c[p] * xc;
            if (im >= 0) s += a0[p] * T(x[p + om]);
            if (ip >= 0) s += a0[p + op] * T(x[p + op]);
            if (jm >= 0) s += a1[p] * T(x[p + ym]);
            if (jp >= 0) s += a1[p + yp] * T(x[p + yp]);
            if (km >= 0) s += a2c * xm;
            if (kp >= 0) s += a2p * xp;
            y[p] = s;
            acc += (double)xc * (double)s;
            xm = xc;
            xc = xp;
            a2c = a2p;
            km = k;
        }
    }
    if (part) {
        const int t = threadIdx.y * blockDim.x + threadIdx.x;
        const int nt = blockDim.x * blockDim.y;
        double v = wave_sum(acc);
        if ((t & 63) == 0) sm[t >> 6] = v;
        __syncthreads();
        if (t == 0) {
            double s = 0.0;
            for (int q = 0; q < (nt + 63) / 64; q++) s += sm[q];
            part[blockIdx.x] = s;
        }
    }
}

// ------------------------------------------------------------------ SpMV, row waves
// Row-wave layout for levels whose rows are long enough: a wave owns one
// x-row segment of 64*CPL cells, CPL consecutive cells per lane, so every
// array is read with one 16-byte load per lane (1 KB per wave instruction).
// The x neighbours come from the neighbouring lanes (lane shuffles) and, at
// the two ends of the segment, from memory. Four waves (rows) per workgroup,
// a z chunk of kc planes per workgroup, y neighbours read directly (they are
// L2 hits: adjacent rows belong to the same or the XCD-neighbouring group).
template <typename T, int CPL>
struct alignas(16) Vec {
    T v[CPL];
};

template <typename T, int CPL>
__device__ __forceinline__ Vec<T, CPL> vld(const T *__restrict__ p) {
    return *reinterpret_cast<const Vec<T, CPL> *>(p);
}

template <typename T, int CPL>
__device__ __forceinline__ Vec<T, CPL> vzero() {
    Vec<T, CPL> r;
#pragma unroll
    for (int e = 0; e < CPL; e++) r.v[e] = T(0);
    return r;
}

// The three stencils that share this layout:
//   RW_APPLY    out = A x, with one FP64 partial of <x, A x> per workgroup
//   RW_RESID    out = f - A x
//   RW_SMOOTH0  first sweep from a zero iterate: with u = f / c, first colour
//               out = u, second colour out = (f - sum_nb a_nb u_nb) / c
// Sums are accumulated in the same order as the tiled kernels.
enum { RW_APPLY = 0, RW_RESID = 1, RW_SMOOTH0 = 2 };

// TX: the type x is stored in (RW_APPLY of the mixed solve: FP32 search
// directions, FP64 operator and product).
template <typename T, int CPL, int MODE, typename TX = T>
__global__ void __launch_bounds__(256) k_stencil_rw(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                    const T *__restrict__ a1, const T *__restrict__ a2,
                                                    const T *__restrict__ f, const TX *__restrict__ x,
                                                    T *__restrict__ y, double *__restrict__ part, int c1, int kc,
                                                    int gx, int gy) {
    __shared__ double sm[4];
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    const int i0 = (bx * 64 + lane) * CPL;
    const int j = by * 4 + w;
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);
    double acc = 0.0;
    typedef Vec<T, CPL> V;
    // the operand at a row/plane offset: x, or u = f / c for the zero-iterate sweep
    auto opnd = [&](int q) -> V {
        if (MODE == RW_SMOOTH0) {
            const V cq = vld<T, CPL>(c + q), fq = vld<T, CPL>(f + q);
            V u;
#pragma unroll
            for (int e = 0; e < CPL; e++) u.v[e] = fq.v[e] / cq.v[e];
            return u;
        } else if constexpr (std::is_same<TX, T>::value) {
            return vld<T, CPL>(x + q);
        } else {
            // CPL narrower values in one load of CPL * sizeof(TX) bytes
            typedef TX xv_t __attribute__((ext_vector_type(CPL)));
            const xv_t t = *reinterpret_cast<const xv_t *>(x + q);
            V r;
#pragma unroll
            for (int e = 0; e < CPL; e++) r.v[e] = T(t[e]);
            return r;
        }
    };
    auto opnd1 = [&](int q) -> T { return MODE == RW_SMOOTH0 ? f[q] / c[q] : T(x[q]); };
    if (i0 < n0 && j < n1 && k0 < k1) {
        const int jm = nbm(j, n1, g.p1), jp = nbp(j, n1, g.p1);
        const int il = nbm(i0, n0, g.p0), ir = nbp(i0 + CPL - 1, n0, g.p0);
        const bool lsh = lane > 0;                    // cell i0-1 is held by lane-1
        const bool rsh = lane < 63 && i0 + CPL < n0;  // cell i0+CPL is held by lane+1
        const bool hasl = lsh || il >= 0, hasr = rsh || ir >= 0;
        const int col = j * n0 + i0;
        const int row0 = j * n0;
        const int dym = (jm - j) * n0, dyp = (jp - j) * n0;
        int km = nbm(k0, n2, g.p2);
        V xm = km >= 0 ? opnd(km * plane + col) : vzero<T, CPL>();
        V xc = opnd(k0 * plane + col);
        V a2c = vld<T, CPL>(a2 + k0 * plane + col);
        for (int k = k0; k < k1; k++) {
            const int p = k * plane + col;
            const int kp = nbp(k, n2, g.p2);
            const V xp = kp >= 0 ? opnd(kp * plane + col) : vzero<T, CPL>();
            const V a2p = kp >= 0 ? vld<T, CPL>(a2 + kp * plane + col) : vzero<T, CPL>();
            const V cc = vld<T, CPL>(c + p), a0c = vld<T, CPL>(a0 + p), a1c = vld<T, CPL>(a1 + p);
            const V xjm = jm >= 0 ? opnd(p + dym) : vzero<T, CPL>();
            const V xjp = jp >= 0 ? opnd(p + dyp) : vzero<T, CPL>();
            const V a1p = jp >= 0 ? vld<T, CPL>(a1 + p + dyp) : vzero<T, CPL>();
            V fc;
            if (MODE != RW_APPLY) fc = vld<T, CPL>(f + p);
            const T xl_s = __shfl(xc.v[CPL - 1], (lane + 63) & 63, 64);
            const T xr_s = __shfl(xc.v[0], (lane + 1) & 63, 64);
            const T ar_s = __shfl(a0c.v[0], (lane + 1) & 63, 64);
            const int rk = k * plane + row0;
            const T xl = lsh ? xl_s : (il >= 0 ? opnd1(rk + il) : T(0));
            const T xr = rsh ? xr_s : (ir >= 0 ? opnd1(rk + ir) : T(0));
            const T ar = rsh ? ar_s : (ir >= 0 ? a0[rk + ir] : T(0));
            V out;
#pragma unroll
            for (int e = 0; e < CPL; e++) {
                const T left = e > 0 ? xc.v[e - 1] : xl;
                const T right = e < CPL - 1 ? xc.v[e + 1] : xr;
                const T aright = e < CPL - 1 ? a0c.v[e + 1] : ar;
                if (MODE == RW_SMOOTH0) {
                    if (((i0 + e + j + k) & 1) == c1) {
                        out.v[e] = xc.v[e];
                    } else {
                        T sum = fc.v[e];
                        if (e > 0 || hasl) sum -= a0c.v[e] * left;
                        if (e < CPL - 1 || hasr) sum -= aright * right;
                        if (jm >= 0) sum -= a1c.v[e] * xjm.v[e];
                        if (jp >= 0) sum -= a1p.v[e] * xjp.v[e];
                        if (km >= 0) sum -= a2c.v[e] * xm.v[e];
                        if (kp >= 0) sum -= a2p.v[e] * xp.v[e];
                        out.v[e] = sum / cc.v[e];
                    }
                } else {
                    T t = cc.v[e] * xc.v[e];
                    if (e > 0 || hasl) t += a0c.v[e] * left;
                    if (e < CPL - 1 || hasr) t += aright * right;
                    if (jm >= 0) t += a1c.v[e] * xjm.v[e];
                    if (jp >= 0) t += a1p.v[e] * xjp.v[e];
                    if (km >= 0) t += a2c.v[e] * xm.v[e];
                    if (kp >= 0) t += a2p.v[e] * xp.v[e];
                    if (MODE == RW_APPLY) {
                        out.v[e] = t;
                        acc += (double)xc.v[e] * (double)t;
                    } else {
                        out.v[e] = fc.v[e] - t;
                    }
                }
            }
            *reinterpret_cast<V *>(y + p) = out;
            xm = xc;
            xc = xp;
            a2c = a2p;
            km = k;
        }
    }
    if (MODE == RW_APPLY && part) {
        double v = wave_sum(acc);
        if (lane == 0) sm[w] = v;
        __syncthreads();
        if (threadIdx.x == 0) part[blockIdx.x] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    }
}

// ------------------------------------------------------------------ stencils from zero
// First symmetric sweep from a zero iterate, as a plain stencil:
//   first colour c1:  v = f / c
//   second colour:    v = (f - sum_nb a_nb f_nb / c_nb) / c
// (the second colour reads the first colour's new values, which are f/c).
template <typename T>
__global__ void __launch_bounds__(256) k_smooth0_t(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                   const T *__restrict__ a1, const T *__restrict__ a2,
                                                   const T *__restrict__ f, T *__restrict__ v, int c1, int kc, int gx, int gy) {
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int i = bx * blockDim.x + threadIdx.x;
    const int j = by * blockDim.y + threadIdx.y;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);
    if (i >= n0 || j >= n1 || k0 >= k1) return;
    const int im = nbm(i, n0, g.p0), ip = nbp(i, n0, g.p0);
    const int jm = nbm(j, n1, g.p1), jp = nbp(j, n1, g.p1);
    const int om = im - i, op = ip - i;
    const int ym = (jm - j) * n0, yp = (jp - j) * n0;
    const int col = j * n0 + i;
    int km = nbm(k0, n2, g.p2);
    // f/c of the own column at k-1, k, k+1 and a2 at k
    T um = km >= 0 ? f[km * plane + col] / c[km * plane + col] : T(0);
    T cc = c[k0 * plane + col];
    T fc = f[k0 * plane + col];
    T a2c = a2[k0 * plane + col];
    for (int k = k0; k < k1; k++) {
        const int p = k * plane + col;
        const int kp = nbp(k, n2, g.p2);
        T cp = T(1), fp = T(0), a2p = T(0);
        if (kp >= 0) {
            cp = c[kp * plane + col];
            fp = f[kp * plane + col];
            a2p = a2[kp * plane + col];
        }
        const T up = kp >= 0 ? fp / cp : T(0);
        T out;
        if (((i + j + k) & 1) == c1) {
            out = fc / cc;
        } else {
            T sum = fc;
            if (im >= 0) sum -= a0[p] * (f[p + om] / c[p + om]);
            if (ip >= 0) sum -= a0[p + op] * (f[p + op] / c[p + op]);
            if (jm >= 0) sum -= a1[p] * (f[p + ym] / c[p + ym]);
            if (jp >= 0) sum -= a1[p + yp] * (f[p + yp] / c[p + yp]);
            if (km >= 0) sum -= a2c * um;
            if (kp >= 0) sum -= a2p * up;
            out = sum / cc;
        }
        v[p] = out;
        um = fc / cc;
        cc = cp;
        fc = fp;
        a2c = a2p;
        km = k;
    }
}

// r = f - A v (the residual handed to the restriction)
template <typename T>
__global__ void __launch_bounds__(256) k_resid_t(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                 const T *__restrict__ a1, const T *__restrict__ a2,
                                                 const T *__restrict__ f, const T *__restrict__ x,
                                                 T *__restrict__ r, int kc, int gx, int gy) {
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int i = bx * blockDim.x + threadIdx.x;
    const int j = by * blockDim.y + threadIdx.y;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);
    if (i >= n0 || j >= n1 || k0 >= k1) return;
    const int im = nbm(i, n0, g.p0), ip = nbp(i, n0, g.p0);
    const int jm = nbm(j, n1, g.p1), jp = nbp(j, n1, g.p1);
    const int om = im - i, op = ip - i;
    const int ym = (jm - j) * n0, yp = (jp - j) * n0;
    const int col = j * n0 + i;
    int km = nbm(k0, n2, g.p2);
    T xm = km >= 0 ? x[km * plane + col] : T(0);
    T xc = x[k0 * plane + col];
    T a2c = a2[k0 * plane + col];
    for (int k = k0; k < k1; k++) {
        const int p = k * plane + col;
        const int kp = nbp(k, n2, g.p2);
        const T xp = kp >= 0 ? x[kp * plane + col] : T(0);
        const T a2p = kp >= 0 ? a2[kp * plane + col] : T(0);
        T t = c[p] * xc;
        if (im >= 0) t += a0[p] * x[p + om];
        if (ip >= 0) t += a0[p + op] * x[p + op];
        if (jm >= 0) t += a1[p] * x[p + ym];
        if (jp >= 0) t += a1[p + yp] * x[p + yp];
        if (km >= 0) t += a2c * xm;
        if (kp >= 0) t += a2p * xp;
        r[p] = f[p] - t;
        xm = xc;
        xc = xp;
        a2c = a2p;
        km = k;
    }
}

// fc = P^T r : one thread per coarse cell. The transfer kernels take their
// multiply-adds explicitly (fma_t) with contraction off, so that the scalar
// and vector forms round alike.
template <typename T, int D>
__global__ void __launch_bounds__(256) k_gather_t(Geo F, Geo C, const T *__restrict__ r, const T *__restrict__ pm,
                                                  const T *__restrict__ pp, T *__restrict__ fc) {
#pragma clang fp contract(off)
    const int I = blockIdx.x * blockDim.x + threadIdx.x;
    const int J = blockIdx.y * blockDim.y + threadIdx.y;
    const int K = blockIdx.z;
    if (I >= C.n0 || J >= C.n1) return;
    const int pc = (K * C.n1 + J) * C.n0 + I;
    const int i = D == 0 ? 2 * I : I, j = D == 1 ? 2 * J : J, k = D == 2 ? 2 * K : K;
    const int e = D == 0 ? i : (D == 1 ? j : k);
    const int nd = D == 0 ? F.n0 : (D == 1 ? F.n1 : F.n2);
    const int per = D == 0 ? F.p0 : (D == 1 ? F.p1 : F.p2);
    const int stride = D == 0 ? 1 : (D == 1 ? F.n0 : F.n0 * F.n1);
    const int pf = (k * F.n1 + j) * F.n0 + i;
    const int l = nbm(e, nd, per);
    T s = r[pf];
    if (e + 1 < nd) s = fma_t(pm[pc], r[pf + stride], s);
    if (l >= 0) {
        const int Jd = D == 0 ? I : (D == 1 ? J : K);
        const int nc = D == 0 ? C.n0 : (D == 1 ? C.n1 : C.n2);
        const int cper = D == 0 ? C.p0 : (D == 1 ? C.p1 : C.p2);
        const int jl = nbm(Jd, nc, cper);
        const int pl = D == 0 ? (K * C.n1 + J) * C.n0 + jl : (D == 1 ? (K * C.n1 + jl) * C.n0 + I
                                                                      : (jl * C.n1 + J) * C.n0 + I);
        s = fma_t(pp[pl], r[pf + (l - e) * stride], s);
    }
    fc[pc] = s;
}

// The same restriction for coarsening in y (D = 1) or z (D = 2) on levels
// whose x rows hold a multiple of CPL cells: x is not coarsened, so CPL
// consecutive coarse cells of a thread sit over CPL consecutive fine cells,
// and every array is read with 16-byte loads. Per cell the arithmetic of
// k_gather_t, in the same order.
template <typename T, int CPL, int D>
__global__ void __launch_bounds__(256) k_gather_v(Geo F, Geo C, const T *__restrict__ r, const T *__restrict__ pm,
                                                  const T *__restrict__ pp, T *__restrict__ fc) {
#pragma clang fp contract(off)
    static_assert(D == 1 || D == 2, "x coarsening has no vector form");
    typedef Vec<T, CPL> V;
    const int I = (blockIdx.x * blockDim.x + threadIdx.x) * CPL;
    const int J = blockIdx.y * blockDim.y + threadIdx.y;
    const int K = blockIdx.z;
    if (I >= C.n0 || J >= C.n1) return;
    const int pc = (K * C.n1 + J) * C.n0 + I;
    const int j = D == 1 ? 2 * J : J, k = D == 2 ? 2 * K : K;
    const int e = D == 1 ? j : k;
    const int nd = D == 1 ? F.n1 : F.n2;
    const int per = D == 1 ? F.p1 : F.p2;
    const int stride = D == 1 ? F.n0 : F.n0 * F.n1;
    const int pf = (k * F.n1 + j) * F.n0 + I;
    const int l = nbm(e, nd, per);
    V s = vld<T, CPL>(r + pf);
    if (e + 1 < nd) {
        const V w = vld<T, CPL>(pm + pc), x = vld<T, CPL>(r + pf + stride);
#pragma unroll
        for (int q = 0; q < CPL; q++) s.v[q] = fma_t(w.v[q], x.v[q], s.v[q]);
    }
    if (l >= 0) {
        const int Jd = D == 1 ? J : K;
        const int jl = nbm(Jd, D == 1 ? C.n1 : C.n2, D == 1 ? C.p1 : C.p2);
        const int pl = D == 1 ? (K * C.n1 + jl) * C.n0 + I : (jl * C.n1 + J) * C.n0 + I;
        const V w = vld<T, CPL>(pp + pl), x = vld<T, CPL>(r + pf + (l - e) * stride);
#pragma unroll
        for (int q = 0; q < CPL; q++) s.v[q] = fma_t(w.v[q], x.v[q], s.v[q]);
    }
    *reinterpret_cast<V *>(fc + pc) = s;
}

// The restriction for coarsening in x on levels whose rows hold a multiple of
// 2 CPL fine cells: CPL coarse cells per thread, their 2 CPL fine residuals
// read with two 16-byte loads, the one fine cell to the left (and its pp
// weight) with scalar loads. Per cell the arithmetic of k_gather_t<T, 0>.
template <typename T, int CPL>
__global__ void __launch_bounds__(256) k_gather_xv(Geo F, Geo C, const T *__restrict__ r, const T *__restrict__ pm,
                                                   const T *__restrict__ pp, T *__restrict__ fc) {
#pragma clang fp contract(off)
    typedef Vec<T, CPL> V;
    const int I0 = (blockIdx.x * blockDim.x + threadIdx.x) * CPL;
    const int J = blockIdx.y * blockDim.y + threadIdx.y;
    const int K = blockIdx.z;
    if (I0 >= C.n0 || J >= C.n1) return;
    const int rowc = (K * C.n1 + J) * C.n0, rowf = (K * F.n1 + J) * F.n0;
    const V r0 = vld<T, CPL>(r + rowf + 2 * I0), r1 = vld<T, CPL>(r + rowf + 2 * I0 + CPL);
    const V w = vld<T, CPL>(pm + rowc + I0), u = vld<T, CPL>(pp + rowc + I0);
    T rr[2 * CPL];
#pragma unroll
    for (int q = 0; q < CPL; q++) {
        rr[q] = r0.v[q];
        rr[CPL + q] = r1.v[q];
    }
    V s;
#pragma unroll
    for (int q = 0; q < CPL; q++) {
        const int I = I0 + q, e = 2 * I;
        T t = rr[2 * q];
        if (e + 1 < F.n0) t = fma_t(w.v[q], rr[2 * q + 1], t);
        const int l = nbm(e, F.n0, F.p0);
        if (l >= 0) {
            T ppl, rl;
            if (q > 0) {
                ppl = u.v[q - 1];
                rl = rr[2 * q - 1];
            } else {
                ppl = pp[rowc + nbm(I, C.n0, C.p0)];
                rl = r[rowf + l];
            }
            t = fma_t(ppl, rl, t);
        }
        s.v[q] = t;
    }
    *reinterpret_cast<V *>(fc + rowc + I0) = s;
}

// ------------------------------------------------------------------ fused sweep
// One symmetric-order Gauss-Seidel sweep, out of place:
//   first colour c1:  v1 = (f - sum a vin) / c        (vin: previous iterate)
//   second colour:    v2 = (f - sum a v1) / c
//   vout = v1 on c1 cells, v2 on the others.
// Identical to the in-place two-pass red/black sweep, since each colour reads
// only the other colour. ZERO_IN: vin == 0 (first sweep of the V-cycle).
// A block covers (SX+2) x (SY+2) cell positions; the outer ring only computes
// first-colour values needed by the core's second colour. The block marches
// over planes s: at step s it computes v1 on plane s+1 and v2 on plane s.
constexpr int SX = 64;

// Workgroup barrier that waits only for LDS traffic, so global loads issued
// for the next plane stay in flight across it (__syncthreads would also drain
// them). gfx9 s_waitcnt: vmcnt = 63, expcnt = 7, lgkmcnt = 0.
__device__ __forceinline__ void lds_barrier() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

template <typename T, bool ZERO_IN, int SY>
__global__ void __launch_bounds__(SX *SY) k_sweep(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                  const T *__restrict__ a1, const T *__restrict__ a2,
                                                  const T *__restrict__ f, const T *__restrict__ vin,
                                                  T *__restrict__ vout, int c1, int kc, int gx, int gy) {
    __shared__ T s_vin[3][SY][SX];
    __shared__ T s_a0[3][SY][SX];
    __shared__ T s_a1[3][SY][SX];
    __shared__ T s_v1[2][SY][SX];
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int iu = bx * (SX - 2) - 1 + tx;
    const int ju = by * (SY - 2) - 1 + ty;
    const int ii = wrapc(iu, n0, g.p0);
    const int jj = wrapc(ju, n1, g.p1);
    const bool valid = ii >= 0 && jj >= 0;
    const int col = valid ? jj * n0 + ii : 0;
    const bool left = tx == 0, right = tx == SX - 1, bot = ty == 0, top = ty == SY - 1;
    const bool corner = (left || right) && (bot || top);
    const bool core = !left && !right && !bot && !top && iu < n0 && ju < n1;
    // the one cell outside the tile a ring position couples to (-1: none)
    int cout = -1;
    if (valid && !corner) {
        if (left) { int q = wrapc(ii - 1, n0, g.p0); cout = q >= 0 ? jj * n0 + q : -1; }
        if (right) { int q = wrapc(ii + 1, n0, g.p0); cout = q >= 0 ? jj * n0 + q : -1; }
        if (bot) { int q = wrapc(jj - 1, n1, g.p1); cout = q >= 0 ? q * n0 + ii : -1; }
        if (top) { int q = wrapc(jj + 1, n1, g.p1); cout = q >= 0 ? q * n0 + ii : -1; }
    }
    // coupling coefficient to that outside cell lives there for +x/+y, here for -x/-y
    const T *__restrict__ aout = right ? a0 : a1;
    const bool out_owns = right || top;
    const int par = (ii + jj) & 1;  // colour of the cell on plane k is (par + k) & 1
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);

    auto kwrap = [&](int k) { return wrapc(k, n2, g.p2); };
    auto ld = [&](const T *__restrict__ a, int kk) -> T { return (valid && kk >= 0) ? a[kk * plane + col] : T(0); };
    auto ldo = [&](const T *__restrict__ a, int kk) -> T { return (cout >= 0 && kk >= 0) ? a[kk * plane + cout] : T(0); };

    int s = k0 - 2;
    // data of plane s+1 (coefficients, vin, outside values) and of plane s+2 (vin, a2)
    int kA = kwrap(s + 1);
    T vin_s = ZERO_IN ? T(0) : ld(vin, kwrap(s));
    T c_A = valid && kA >= 0 ? c[kA * plane + col] : T(1);
    T f_A = ld(f, kA), a0_A = ld(a0, kA), a1_A = ld(a1, kA), a2_A = ld(a2, kA);
    T vin_A = ZERO_IN ? T(0) : ld(vin, kA);
    T vo_A = ZERO_IN ? T(0) : ldo(vin, kA);
    T ao_A = out_owns ? ldo(aout, kA) : T(0);
    int kB = kwrap(s + 2);
    T vin_B = ZERO_IN ? T(0) : ld(vin, kB);
    T a2_B = ld(a2, kB);
    T c_s = T(1), f_s = T(0), a0_s = T(0), a1_s = T(0), a2_s = T(0);
    T v1_m = T(0), v1_0 = T(0);
    int slot3 = 0;  // slot of plane s+1 in the 3-deep ring
    for (; s < k1; s++) {
        // prefetch: plane s+2 coefficients and outside values, plane s+3 vin and a2
        const int kN = kwrap(s + 2), kN2 = kwrap(s + 3);
        const T c_N = valid && kN >= 0 ? c[kN * plane + col] : T(1);
        const T f_N = ld(f, kN), a0_N = ld(a0, kN), a1_N = ld(a1, kN);
        const T vo_N = ZERO_IN ? T(0) : ldo(vin, kN);
        const T ao_N = out_owns ? ldo(aout, kN) : T(0);
        const T vin_N2 = ZERO_IN ? T(0) : ld(vin, kN2);
        const T a2_N2 = ld(a2, kN2);
        // publish plane s+1
        if (!ZERO_IN) s_vin[slot3][ty][tx] = vin_A;
        s_a0[slot3][ty][tx] = a0_A;
        s_a1[slot3][ty][tx] = a1_A;
        lds_barrier();
        const int ks = kwrap(s);
        // first colour on plane s+1
        T v1_p = T(0);
        if (valid && kA >= 0 && !corner && ((par + kA) & 1) == c1) {
            T sum = f_A;
            if (!ZERO_IN) {
                const T xm = left ? vo_A : s_vin[slot3][ty][tx - 1];
                const T xp = right ? vo_A : s_vin[slot3][ty][tx + 1];
                const T ym = bot ? vo_A : s_vin[slot3][ty - 1][tx];
                const T yp = top ? vo_A : s_vin[slot3][ty + 1][tx];
                const T a0p = right ? ao_A : s_a0[slot3][ty][tx + 1];
                const T a1p = top ? ao_A : s_a1[slot3][ty + 1][tx];
                sum -= a0_A * xm;
                sum -= a0p * xp;
                sum -= a1_A * ym;
                sum -= a1p * yp;
                sum -= a2_A * vin_s;
                sum -= a2_B * vin_B;
            }
            v1_p = sum / c_A;
        }
        s_v1[(s + 1) & 1][ty][tx] = v1_p;
        // second colour on plane s (core only)
        if (s >= k0 && core && ks >= 0) {
            T out;
            if (((par + ks) & 1) == c1) {
                out = v1_0;
            } else {
                const int sl = (slot3 + 2) % 3;  // slot of plane s
                T sum = f_s;
                sum -= a0_s * s_v1[s & 1][ty][tx - 1];
                sum -= s_a0[sl][ty][tx + 1] * s_v1[s & 1][ty][tx + 1];
                sum -= a1_s * s_v1[s & 1][ty - 1][tx];
                sum -= s_a1[sl][ty + 1][tx] * s_v1[s & 1][ty + 1][tx];
                sum -= a2_s * v1_m;
                sum -= a2_A * v1_p;
                out = sum / c_s;
            }
            vout[ks * plane + col] = out;
        }
        // rotate: plane s+1 -> s, prefetched plane s+2 -> s+1
        vin_s = vin_A;
        c_s = c_A;
        f_s = f_A;
        a0_s = a0_A;
        a1_s = a1_A;
        a2_s = a2_A;
        kA = kN;
        c_A = c_N;
        f_A = f_N;
        a0_A = a0_N;
        a1_A = a1_N;
        a2_A = a2_B;
        vin_A = vin_B;
        vo_A = vo_N;
        ao_A = ao_N;
        vin_B = vin_N2;
        a2_B = a2_N2;
        v1_m = v1_0;
        v1_0 = v1_p;
        slot3 = (slot3 + 1) % 3;
    }
}

// ------------------------------------------------------------------ sweep over whole rows
// The sweep of k_sweep on levels whose x rows fit one workgroup row
// (n0 <= NX, NX = 32, 64 or 128): a workgroup of NX x NY threads (NX NY =
// 1024) holds whole rows, so every x neighbour is in the tile (across the row
// end for periodic x) and only y has a recompute ring (NY - 2 output rows).
// On 128-cell rows k_sweep's 62-column tiles need three tile columns per row
// and half of the threads do no output; here a quarter do none. Per cell the
// arithmetic of k_sweep in the same order; a neighbour beyond a wall
// contributes 0 * 0 there and here, so the two kernels are bit-identical.
template <typename T, bool ZERO_IN, int NX>
__global__ void __launch_bounds__(1024) k_sweep_row(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                    const T *__restrict__ a1, const T *__restrict__ a2,
                                                    const T *__restrict__ f, const T *__restrict__ vin,
                                                    T *__restrict__ vout, int c1, int kc, int gy) {
    constexpr int NY = 1024 / NX;
    __shared__ T s_vin[3][NY][NX];
    __shared__ T s_a0[3][NY][NX];
    __shared__ T s_a1[3][NY][NX];
    __shared__ T s_v1[2][NY][NX];
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    int bx, by, bz;
    tile_of(1, gy, bx, by, bz);
    const int ju = by * (NY - 2) - 1 + ty;
    const int jj = wrapc(ju, n1, g.p1);
    const bool inrow = tx < n0;  // lanes past the row end hold zeros
    const bool valid = inrow && jj >= 0;
    const int col = valid ? jj * n0 + tx : 0;
    // in-row neighbours in the tile (-1: beyond a wall, or a lane past the row)
    const int txm = inrow ? nbm(tx, n0, g.p0) : -1;
    const int txp = inrow ? nbp(tx, n0, g.p0) : -1;
    const bool bot = ty == 0, top = ty == NY - 1;
    const bool core = !bot && !top && ju < n1 && inrow;
    // the one cell outside the tile a ring row couples to (-1: none)
    int cout = -1;
    if (valid) {
        if (bot) { int q = wrapc(jj - 1, n1, g.p1); cout = q >= 0 ? q * n0 + tx : -1; }
        if (top) { int q = wrapc(jj + 1, n1, g.p1); cout = q >= 0 ? q * n0 + tx : -1; }
    }
    const int par = (tx + jj) & 1;  // colour of the cell on plane k is (par + k) & 1
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);

    auto kwrap = [&](int k) { return wrapc(k, n2, g.p2); };
    auto ld = [&](const T *__restrict__ a, int kk) -> T { return (valid && kk >= 0) ? a[kk * plane + col] : T(0); };
    auto ldo = [&](const T *__restrict__ a, int kk) -> T { return (cout >= 0 && kk >= 0) ? a[kk * plane + cout] : T(0); };
    // an x neighbour's entry of an LDS plane (0 beyond a wall)
    auto lx = [&](const T (*S)[NX], int q) -> T { return q >= 0 ? S[ty][q] : T(0); };

    int s = k0 - 2;
    int kA = kwrap(s + 1);
    T vin_s = ZERO_IN ? T(0) : ld(vin, kwrap(s));
    T c_A = valid && kA >= 0 ? c[kA * plane + col] : T(1);
    T f_A = ld(f, kA), a0_A = ld(a0, kA), a1_A = ld(a1, kA), a2_A = ld(a2, kA);
    T vin_A = ZERO_IN ? T(0) : ld(vin, kA);
    T vo_A = ZERO_IN ? T(0) : ldo(vin, kA);
    T ao_A = top ? ldo(a1, kA) : T(0);
    int kB = kwrap(s + 2);
    T vin_B = ZERO_IN ? T(0) : ld(vin, kB);
    T a2_B = ld(a2, kB);
    T c_s = T(1), f_s = T(0), a0_s = T(0), a1_s = T(0), a2_s = T(0);
    T v1_m = T(0), v1_0 = T(0);
    int slot3 = 0;
    for (; s < k1; s++) {
        const int kN = kwrap(s + 2), kN2 = kwrap(s + 3);
        const T c_N = valid && kN >= 0 ? c[kN * plane + col] : T(1);
        const T f_N = ld(f, kN), a0_N = ld(a0, kN), a1_N = ld(a1, kN);
        const T vo_N = ZERO_IN ? T(0) : ldo(vin, kN);
        const T ao_N = top ? ldo(a1, kN) : T(0);
        const T vin_N2 = ZERO_IN ? T(0) : ld(vin, kN2);
        const T a2_N2 = ld(a2, kN2);
        if (!ZERO_IN) s_vin[slot3][ty][tx] = vin_A;
        s_a0[slot3][ty][tx] = a0_A;
        s_a1[slot3][ty][tx] = a1_A;
        lds_barrier();
        const int ks = kwrap(s);
        // first colour on plane s+1 (ring rows included)
        T v1_p = T(0);
        if (valid && kA >= 0 && ((par + kA) & 1) == c1) {
            T sum = f_A;
            if (!ZERO_IN) {
                const T xm = lx(s_vin[slot3], txm);
                const T xp = lx(s_vin[slot3], txp);
                const T ym = bot ? vo_A : s_vin[slot3][ty - 1][tx];
                const T yp = top ? vo_A : s_vin[slot3][ty + 1][tx];
                const T a0p = lx(s_a0[slot3], txp);
                const T a1p = top ? ao_A : s_a1[slot3][ty + 1][tx];
                sum -= a0_A * xm;
                sum -= a0p * xp;
                sum -= a1_A * ym;
                sum -= a1p * yp;
                sum -= a2_A * vin_s;
                sum -= a2_B * vin_B;
            }
            v1_p = sum / c_A;
        }
        s_v1[(s + 1) & 1][ty][tx] = v1_p;
        // second colour on plane s (core rows only)
        if (s >= k0 && core && ks >= 0) {
            T out;
            if (((par + ks) & 1) == c1) {
                out = v1_0;
            } else {
                const int sl = (slot3 + 2) % 3;
                T sum = f_s;
                sum -= a0_s * lx(s_v1[s & 1], txm);
                sum -= lx(s_a0[sl], txp) * lx(s_v1[s & 1], txp);
                sum -= a1_s * s_v1[s & 1][ty - 1][tx];
                sum -= s_a1[sl][ty + 1][tx] * s_v1[s & 1][ty + 1][tx];
                sum -= a2_s * v1_m;
                sum -= a2_A * v1_p;
                out = sum / c_s;
            }
            vout[ks * plane + col] = out;
        }
        vin_s = vin_A;
        c_s = c_A;
        f_s = f_A;
        a0_s = a0_A;
        a1_s = a1_A;
        a2_s = a2_A;
        kA = kN;
        c_A = c_N;
        f_A = f_N;
        a0_A = a0_N;
        a1_A = a1_N;
        a2_A = a2_B;
        vin_A = vin_B;
        vo_A = vo_N;
        ao_A = ao_N;
        vin_B = vin_N2;
        a2_B = a2_N2;
        v1_m = v1_0;
        v1_0 = v1_p;
        slot3 = (slot3 + 1) % 3;
    }
}

// ------------------------------------------------------------------ two fused sweeps
// Two consecutive sweeps of the same colour order c1 (the post-smoothing of a
// V(., 2) cycle) in one launch: four colour half-steps
//   h1: colour c1   from vin       h2: colour c2 from h1
//   h3: colour c1   from h2        h4: colour c2 from h3
// vout = h3 on c1 cells, h4 on c2 cells: the result of two k_sweep launches,
// with the same arithmetic in the same order, so bit-identical to them.
// A 64 x 16 workgroup recomputes a 3-cell ring (output core 58 x 10): h1 runs
// on every position (the outer ring reads the cells just outside the tile),
// h2 from depth 1, h3 from depth 2, h4 on the core. The planes are pipelined:
// at step s, h1 on plane s+3, h2 on s+2, h3 on s+1, h4 on s. Each field
// lives in LDS for the in-plane neighbours of the next half-step and in
// registers (three planes) for its z neighbours; a_x, a_y are in LDS for the
// four planes in use. One LDS barrier per step.
constexpr int R2 = 3;  // recompute ring of the fused pair

// ZERO_IN: vin == 0 (the first two sweeps of the pre-smoothing): h1 is f / c,
// vin is never read, and the pair equals the zero-iterate sweep followed by a
// sweep of the same order.
template <typename T, int SY, bool ZERO_IN = false>
__global__ void __launch_bounds__(SX *SY) k_sweep2(Geo g, const T *__restrict__ c, const T *__restrict__ a0,
                                                   const T *__restrict__ a1, const T *__restrict__ a2,
                                                   const T *__restrict__ f, const T *__restrict__ vin,
                                                   T *__restrict__ vout, int c1, int kc, int gx, int gy) {
    __shared__ T s_vin[2][SY][SX];
    __shared__ T s_a0[5][SY][SX];
    __shared__ T s_a1[5][SY][SX];
    __shared__ T s_h[3][2][SY][SX];  // fields h1, h2, h3, two planes each
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int n0 = g.n0, n1 = g.n1, n2 = g.n2;
    const int plane = n0 * n1;
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int iu = bx * (SX - 2 * R2) - R2 + tx;
    const int ju = by * (SY - 2 * R2) - R2 + ty;
    const int ii = wrapc(iu, n0, g.p0);
    const int jj = wrapc(ju, n1, g.p1);
    const bool valid = ii >= 0 && jj >= 0;
    const int col = valid ? jj * n0 + ii : 0;
    const int depth = min(min(tx, SX - 1 - tx), min(ty, SY - 1 - ty));
    const bool left = tx == 0, right = tx == SX - 1, bot = ty == 0, top = ty == SY - 1;
    const bool corner = (left || right) && (bot || top);
    const bool core = depth >= R2 && iu < n0 && ju < n1;
    int cout = -1;
    if (valid && !corner) {
        if (left) { int q = wrapc(ii - 1, n0, g.p0); cout = q >= 0 ? jj * n0 + q : -1; }
        if (right) { int q = wrapc(ii + 1, n0, g.p0); cout = q >= 0 ? jj * n0 + q : -1; }
        if (bot) { int q = wrapc(jj - 1, n1, g.p1); cout = q >= 0 ? q * n0 + ii : -1; }
        if (top) { int q = wrapc(jj + 1, n1, g.p1); cout = q >= 0 ? q * n0 + ii : -1; }
    }
    const T *__restrict__ aout = right ? a0 : a1;
    const bool out_owns = right || top;
    const int par = (ii + jj) & 1;
    const int c2 = c1 ^ 1;
    const int k0 = bz * kc;
    const int k1 = min(n2, k0 + kc);

    auto kwrap = [&](int k) { return wrapc(k, n2, g.p2); };
    auto ld = [&](const T *__restrict__ a, int kk) -> T { return (valid && kk >= 0) ? a[kk * plane + col] : T(0); };
    auto ldo = [&](const T *__restrict__ a, int kk) -> T { return (cout >= 0 && kk >= 0) ? a[kk * plane + cout] : T(0); };
    auto ldc = [&](int kk) -> T { return valid && kk >= 0 ? c[kk * plane + col] : T(1); };
    // colour of this cell on (unwrapped) plane k, from its wrapped index
    auto colour = [&](int kk) { return (par + kk) & 1; };

    // registers: index 0 = plane P = s+3 (h1's plane), 1 = P-1, 2 = P-2, 3 = P-3
    T cq[4], fq[4];
    T a2q[5];        // a2 of planes P+1, P, P-1, P-2, P-3
    T vin_m, vin_p;  // vin of planes P-1 and P+1
    // the fields' values on the two planes below the one computed this step:
    // h1 of P-1, P-2; h2 of P-2, P-3; h3 of P-3, P-4
    T h1[2], h2[2], h3[2];
    // data of plane P for the first step
    int s = k0 - 6;
    int kP = kwrap(s + 3);
    for (int q = 0; q < 4; q++) {
        const int kq = kwrap(s + 3 - q);
        cq[q] = ldc(kq);
        fq[q] = ld(f, kq);
    }
    for (int q = 0; q < 5; q++) a2q[q] = ld(a2, kwrap(s + 4 - q));
    vin_m = ZERO_IN ? T(0) : ld(vin, kwrap(s + 2));
    vin_p = ZERO_IN ? T(0) : ld(vin, kwrap(s + 4));
    T vin_P = ZERO_IN ? T(0) : ld(vin, kP), a0_P = ld(a0, kP), a1_P = ld(a1, kP);
    T vo_P = ZERO_IN ? T(0) : ldo(vin, kP), ao_P = out_owns ? ldo(aout, kP) : T(0);
    for (int q = 0; q < 2; q++) h1[q] = h2[q] = h3[q] = T(0);
    int sa = 0;  // slot of plane P in the 5-deep a0/a1 ring
    for (; s < k1; s++) {
        const int P = s + 3;
        // prefetch plane P+1 (and vin, a2 of P+2)
        const int kN = kwrap(P + 1), kN2 = kwrap(P + 2);
        const T c_N = ldc(kN), f_N = ld(f, kN), a0_N = ld(a0, kN), a1_N = ld(a1, kN);
        const T vo_N = ZERO_IN ? T(0) : ldo(vin, kN), ao_N = out_owns ? ldo(aout, kN) : T(0);
        const T vin_N2 = ZERO_IN ? T(0) : ld(vin, kN2), a2_N2 = ld(a2, kN2);
        // publish plane P
        const int sv = P & 1;
        if (!ZERO_IN) s_vin[sv][ty][tx] = vin_P;
        s_a0[sa][ty][tx] = a0_P;
        s_a1[sa][ty][tx] = a1_P;
        lds_barrier();
        const int sa1 = sa == 0 ? 4 : sa - 1, sa2 = sa1 == 0 ? 4 : sa1 - 1, sa3 = sa2 == 0 ? 4 : sa2 - 1;
        // one half-step at plane p (ring slot sl of a_x, a_y): in-plane neighbours
        // from field slab F, z neighbours zm / zp, couplings a2 below / above
        auto half = [&](int q, int sl, const T (*F)[SX], T zm, T zp, T a2m, T a2p, bool ring) -> T {
            T sum = fq[q];
            const T a0s = s_a0[sl][ty][tx], a1s = s_a1[sl][ty][tx];
            const T xm = (ring && left) ? vo_P : F[ty][tx - 1];
            const T xp = (ring && right) ? vo_P : F[ty][tx + 1];
            const T ym = (ring && bot) ? vo_P : F[ty - 1][tx];
            const T yp = (ring && top) ? vo_P : F[ty + 1][tx];
            const T a0p = (ring && right) ? ao_P : s_a0[sl][ty][tx + 1];
            const T a1p = (ring && top) ? ao_P : s_a1[sl][ty + 1][tx];
            sum -= a0s * xm;
            sum -= a0p * xp;
            sum -= a1s * ym;
            sum -= a1p * yp;
            sum -= a2m * zm;
            sum -= a2p * zp;
            return sum / cq[q];
        };
        // h1 on P (every position but the corners; the outer ring reads outside values)
        T n1v = T(0);
        if (valid && kP >= 0 && !corner && colour(kP) == c1)
            n1v = ZERO_IN ? fq[0] / cq[0] : half(0, sa, s_vin[sv], vin_m, vin_p, a2q[1], a2q[0], true);
        // h2 on P-1 from h1 (depth >= 1)
        const int k_1 = kwrap(P - 1);
        T n2v = T(0);
        if (valid && k_1 >= 0 && depth >= 1 && colour(k_1) == c2)
            n2v = half(1, sa1, s_h[0][(P - 1) & 1], h1[1], n1v, a2q[2], a2q[1], false);
        // h3 on P-2 from h2 (depth >= 2)
        const int k_2 = kwrap(P - 2);
        T n3v = T(0);
        if (valid && k_2 >= 0 && depth >= 2 && colour(k_2) == c1)
            n3v = half(2, sa2, s_h[1][(P - 2) & 1], h2[1], n2v, a2q[3], a2q[2], false);
        // h4 on P-3 = s from h3, stored on the core
        const int ks = kwrap(s);
        if (s >= k0 && core && ks >= 0) {
            T out;
            if (colour(ks) == c1) {
                out = h3[0];
            } else {
                out = half(3, sa3, s_h[2][s & 1], h3[1], n3v, a2q[4], a2q[3], false);
            }
            vout[ks * plane + col] = out;
        }
        // publish the new field planes (read at the next step, after its barrier)
        s_h[0][P & 1][ty][tx] = n1v;
        s_h[1][(P - 1) & 1][ty][tx] = n2v;
        s_h[2][(P - 2) & 1][ty][tx] = n3v;
        // rotate: plane P+1 becomes P
        h3[1] = h3[0];
        h3[0] = n3v;
        h2[1] = h2[0];
        h2[0] = n2v;
        h1[1] = h1[0];
        h1[0] = n1v;
        for (int q = 3; q > 0; q--) {
            cq[q] = cq[q - 1];
            fq[q] = fq[q - 1];
        }
        cq[0] = c_N;
        fq[0] = f_N;
        for (int q = 4; q > 0; q--) a2q[q] = a2q[q - 1];
        a2q[0] = a2_N2;
        vin_m = vin_P;
        vin_P = vin_p;
        vin_p = vin_N2;
        a0_P = a0_N;
        a1_P = a1_N;
        vo_P = vo_N;
        ao_P = ao_N;
        kP = kN;
        sa = sa == 4 ? 0 : sa + 1;
    }
}

// ------------------------------------------------------------------ transfers over skipped levels
// Three transfers along three directions in one launch, between a level and the
// third one below it when the two levels between are not smoothed (full
// coarsening): neither is stored. DA, DB, DC: the directions in the order of the
// coarsening. One thread per cell of the lowest level; per value the operations
// of k_gather_t and k_prolong_t, so the same bits as three launches.
// Bound by the latency of the loads and, on large levels, by the intermediate
// levels' passes that it saves: all loads are unconditional (a value that is not
// there repeats another and is left out by a select), since behind branches they
// ran one after the other (13.2 us a restriction). FP64, mean of the cycle's
// chains on 128^3: three restrictions 11.6 -> 9.9 us, three prolongations 13.7 ->
// 11.1 us; on 64^3 9.2 -> 4.6 and 13.3 -> 6.5 us.
template <typename T>
struct Chain {
    Geo g[4];                   // the level and the three below
    const T *pm[3], *pp[3];     // weights, stored on levels 1, 2, 3
};

template <int DA, int DB>
__device__ __forceinline__ int at_abc(const Geo &g, int a, int b, int c) {
    const int x = DA == 0 ? a : (DB == 0 ? b : c), y = DA == 1 ? a : (DB == 1 ? b : c),
              z = DA == 2 ? a : (DB == 2 ? b : c);
    return (z * g.n1 + y) * g.n0 + x;
}
template <int D>
__device__ __forceinline__ int len(const Geo &g) {
    return D == 0 ? g.n0 : (D == 1 ? g.n1 : g.n2);
}
template <int D>
__device__ __forceinline__ int per(const Geo &g) {
    return D == 0 ? g.p0 : (D == 1 ? g.p1 : g.p2);
}

// P^T along one direction at coarse position e: v(fine position), the weights'
// values through w(positions on the coarse level)
template <int D, typename T, typename V, typename W>
__device__ __forceinline__ T gather1(const Geo &F, const Geo &C, int e, const T *pm, const T *pp, V v, W w) {
#pragma clang fp contract(off)
    const int n = len<D>(F), l = nbm(2 * e, n, per<D>(F)), el = nbm(e, len<D>(C), per<D>(C));
    const bool odd = 2 * e + 1 < n;
    const T v0 = v(2 * e), v1 = v(odd ? 2 * e + 1 : 2 * e), vl = v(l >= 0 ? l : 2 * e);
    const T w0 = pm[w(e)], wl = pp[w(el >= 0 ? el : e)];
    T s = v0;
    s = odd ? fma_t(w0, v1, s) : s;
    s = l >= 0 ? fma_t(wl, vl, s) : s;
    return s;
}

template <typename T, int DA, int DB, int DC>
__global__ void __launch_bounds__(256) k_gather3(Chain<T> ch, const T *__restrict__ r, T *__restrict__ fc) {
    const Geo g0 = ch.g[0], g1 = ch.g[1], g2 = ch.g[2], g3 = ch.g[3];
    const T *__restrict__ m1 = ch.pm[0], *__restrict__ p1 = ch.pp[0], *__restrict__ m2 = ch.pm[1],
            *__restrict__ p2 = ch.pp[1], *__restrict__ m3 = ch.pm[2], *__restrict__ p3 = ch.pp[2];
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y * blockDim.y + threadIdx.y, z = blockIdx.z;
    if (x >= g3.n0 || y >= g3.n1) return;
    const int A = DA == 0 ? x : (DA == 1 ? y : z), B = DB == 0 ? x : (DB == 1 ? y : z),
              C = DC == 0 ? x : (DC == 1 ? y : z);
    auto v1 = [&](int b, int c) {
        return gather1<DA>(
            g0, g1, A, m1, p1, [&](int a) { return r[at_abc<DA, DB>(g0, a, b, c)]; },
            [&](int a) { return at_abc<DA, DB>(g1, a, b, c); });
    };
    auto v2 = [&](int c) {
        return gather1<DB>(
            g1, g2, B, m2, p2, [&](int b) { return v1(b, c); }, [&](int b) { return at_abc<DA, DB>(g2, A, b, c); });
    };
    fc[(z * g3.n1 + y) * g3.n0 + x] = gather1<DC>(
        g2, g3, C, m3, p3, [&](int c) { return v2(c); }, [&](int c) { return at_abc<DA, DB>(g3, A, B, c); });
}

// the odd fine value between two coarse ones (i: the weights' index; right: there is
// a second one)
template <typename T>
__device__ __forceinline__ T between(const T *pm, const T *pp, int i, T v0, T v1, bool right) {
#pragma clang fp contract(off)
    const T wm = pm[i], wp = pp[i], add = wm * v0;
    return right ? fma_t(wp, v1, add) : add;
}

// vin == nullptr: vout = P v_c
template <typename T, int DA, int DB, int DC>
__global__ void __launch_bounds__(256) k_prolong3(Chain<T> ch, const T *__restrict__ vc, const T *vin, T *vout) {
#pragma clang fp contract(off)
    const Geo g0 = ch.g[0], g1 = ch.g[1], g2 = ch.g[2], g3 = ch.g[3];
    const T *__restrict__ m1 = ch.pm[0], *__restrict__ p1 = ch.pp[0], *__restrict__ m2 = ch.pm[1],
            *__restrict__ p2 = ch.pp[1], *__restrict__ m3 = ch.pm[2], *__restrict__ p3 = ch.pp[2];
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y * blockDim.y + threadIdx.y, z = blockIdx.z;
    if (x >= g3.n0 || y >= g3.n1) return;
    const int A = DA == 0 ? x : (DA == 1 ? y : z), B = DB == 0 ? x : (DB == 1 ? y : z),
              C = DC == 0 ? x : (DC == 1 ? y : z);
    const int A1 = nbp(A, len<DA>(g3), per<DA>(g3)), B1 = nbp(B, len<DB>(g3), per<DB>(g3)),
              C1 = nbp(C, len<DC>(g3), per<DC>(g3));
    const bool ra = A1 >= 0, rb = B1 >= 0, rc = C1 >= 0;
    const bool oa = 2 * A + 1 < len<DA>(g0), ob = 2 * B + 1 < len<DB>(g0), oc = 2 * C + 1 < len<DC>(g0);
    const int a_[2] = {A, ra ? A1 : A}, b_[2] = {B, rb ? B1 : B};
    const int c1 = rc ? C1 : C;
    // along DC: level 2 at (a_, b_, 2C + 0, 1); a skipped level's value is 0 + P v
    T t2[2][2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int at = at_abc<DA, DB>(g3, a_[i], b_[j], C);
            const T u0 = vc[at], u1 = vc[at_abc<DA, DB>(g3, a_[i], b_[j], c1)];
            t2[i][j][0] = T(0) + u0;
            t2[i][j][1] = T(0) + between(m3, p3, at, u0, u1, rc);
        }
    // along DB: level 1 at (a_, 2B + 0, 1, 2C + 0, 1)
    T t1[2][2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            t1[i][0][k] = T(0) + t2[i][0][k];
            t1[i][1][k] = T(0) + between(m2, p2, at_abc<DA, DB>(g2, a_[i], B, k && oc ? 2 * C + 1 : 2 * C), t2[i][0][k],
                                         t2[i][1][k], rb);
        }
    // along DA: this level (a cell past an odd end repeats the one before it)
    T o[2][2][2], w[2][2][2];
    int ao[2][2][2];
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int fb = j && ob ? 2 * B + 1 : 2 * B, fc = k && oc ? 2 * C + 1 : 2 * C;
            ao[0][j][k] = at_abc<DA, DB>(g0, 2 * A, fb, fc);
            ao[1][j][k] = at_abc<DA, DB>(g0, oa ? 2 * A + 1 : 2 * A, fb, fc);
            o[0][j][k] = t1[0][j][k];
            o[1][j][k] = between(m1, p1, at_abc<DA, DB>(g1, A, fb, fc), t1[0][j][k], t1[1][j][k], ra);
#pragma unroll
            for (int i = 0; i < 2; i++) w[i][j][k] = vin ? vin[ao[i][j][k]] : T(0);
        }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int i = 0; i < 2; i++)
                if ((!i || oa) && (!j || ob) && (!k || oc)) vout[ao[i][j][k]] = w[i][j][k] + o[i][j][k];
}

// ------------------------------------------------------------------ the pair, two cells per lane
// The pair of k_sweep2 in FP32 on levels of an even row length. In k_sweep2 a
// lane holds one cell column and half of the lanes idle: at the step whose
// newest plane is P, h1 on P, h2 on P-1, h3 on P-2 and h4 on P-3 all fall on
// the columns of one x-y parity, and on the others' at the next step. Its
// vector instructions alone took 156 of the 247 us of a 256^3 launch. Here a
// lane holds both columns of an x pair, A and B; at every step one of them (X)
// does all four half-steps and the other (Y) none, so no lane idles.
// - In-plane x neighbours: the other column's values of the previous step, its
//   own (a register) and the adjacent lane's (a lane shift; no LDS).
// - y neighbours and a_y through LDS, one value per pair and field (the field
//   exists on one colour only): 80 KB.
// - A tile is 64 x 32 cells: 16 waves, wave w holding rows w and w + 16 (equal
//   parity, so that which of the pair is A is the same for the whole wave and a
//   template argument, S = its x parity). The ring is 4 cells wide, so the
//   outermost cells only hand on vin and nothing outside the tile is read:
//   output core 56 x 24.
// - No cell is masked: outside a wall f, a are 0 and c is 1, which gives 0, and
//   what the tile's outermost cells compute from neighbours they do not have
//   stays inside the ring.
// - Loads are issued two planes ahead, each of an x pair (8 bytes) and all of
//   them unconditional: buffer loads, whose offsets past the plane give 0 (and
//   whose stores there are dropped). Behind branches the wait for the planes of
//   the last step became a wait for those just issued (215 us).
// - Six steps per loop iteration: the life of a loaded value, so that the queues
//   shift by renaming (a copy of a load in flight waits for it), and of the
//   LDS slots, so that their addresses are constants.
// Bound by the traffic of the tiles with their rings: 657 MB a launch by the
// counters (1.4 times the arrays) at 4.6 TB/s. Per cell the operations and
// roundings of k_sweep2, so bit-identical to it. In a 256^3 solve 247 -> 145 us,
// from zero 209 -> 142 us.
constexpr int PX = 64, PY = 32, PR = 4;
static_assert(PX - 2 * PR == PAIR_CX && PY - 2 * PR == PAIR_CY, "pair_form counts these tiles");
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float lane_down(float v) {  // from lane - 1
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_up(float v) {  // from lane + 1
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}

struct PairLds {
    float a1[6][2][PY][PX / 2];  // a_y of six planes, even and odd cells
    float h[3][2][PY][PX / 2];   // fields h1, h2, h3, two planes
    float v[2][PY][PX / 2];      // vin of two planes (the second colour's cells)
};

template <bool ZERO_IN, int S>
__device__ __forceinline__ void pair_march(PairLds &M, const Geo &g, const float *__restrict__ c,
                                           const float *__restrict__ a0, const float *__restrict__ a1,
                                           const float *__restrict__ a2, const float *__restrict__ f,
                                           const float *__restrict__ vin, float *__restrict__ vout, int k0, int k1,
                                           int ty, int q, bool valid, unsigned oE, unsigned oS) {
#pragma clang fp contract(off)
    const int n2 = g.n2, per2 = g.p2;
    const long long plane = (long long)g.n0 * g.n1;
    const unsigned bytes = 4u * (unsigned)plane;
    // the pair at element offset o (a plane's first); zero outside the plane's
    // bytes and for n == 0
    auto at2 = [&](const float *p, long long o, unsigned n) -> f32x2 {
        __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(p + o), 0, (int)n, 0x00027000);
        return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)oE, 0, 0));
    };
    // c, f, a0 of planes P+2 .. P-3, a1 of P+2 .. P, a2 of P+2 .. P-3 and P+3's at
    // the end of a step, of both columns; vin of the second colour's, P+3 .. P-1
    f32x2 cq[6], fq[6], a0q[6], a1q[3], a2q[7];
    float w[5];
#pragma unroll
    for (int i = 0; i < 6; i++) {
        cq[i] = f32x2{1.0f, 1.0f};
        fq[i] = a0q[i] = f32x2{0.0f, 0.0f};
    }
#pragma unroll
    for (int i = 0; i < 7; i++) a2q[i] = f32x2{0.0f, 0.0f};
    a1q[2] = f32x2{0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 5; i++) w[i] = 0.0f;
    float h1[2] = {0.0f, 0.0f}, h2[2] = {0.0f, 0.0f}, h3[2] = {0.0f, 0.0f};  // of the last two steps
    int P = k0 - 3;
    // before the first step, queues as the step's shift expects them: planes P+1,
    // P of c, f, a0, a1 and P+2 .. P of a2, P+2 .. P-1 of vin. The column active
    // at plane P is A, so the second colour's is B there and at P+2.
#pragma unroll
    for (int i = 3; i >= 0; i--) {
        const int kk = wrapc(P + 2 - i, n2, per2);
        const long long o = kk < 0 ? 0 : kk * plane;
        const unsigned n = kk < 0 ? 0 : bytes;
        if (i == 1 || i == 2) {
            cq[i - 1] = at2(c, o, n);
            fq[i - 1] = at2(f, o, n);
            a0q[i - 1] = at2(a0, o, n);
            a1q[i - 1] = at2(a1, o, n);
        }
        if (i < 3) a2q[i] = at2(a2, o, n);
        if (!ZERO_IN) w[i] = at2(vin, o, n)[(i & 1) ? S : 1 - S];
    }
    // planes P + 2 and P + 3: element offset and bytes (0 outside a wall)
    int kM = per2 ? wrapc(P + 3, n2, 1) : P + 3;
    const int kN = wrapc(P + 2, n2, per2);
    long long oN = kN * plane, oM = kM * plane;
    unsigned nN = kN < 0 ? 0 : bytes;
    const unsigned out = valid ? 0u : 0x40000000u;
    // one step; m: its number modulo 6, even where column A is active
    auto step = [&](auto mc) {
        constexpr int m = decltype(mc)::value, X = m & 1, Y = 1 - X, x = X ^ S, y = 1 - x;  // x: the active cell's parity
        const bool ok = (unsigned)(per2 ? 0 : P) + out < (unsigned)n2;
#pragma unroll
        for (int i = 5; i > 0; i--) {
            cq[i] = cq[i - 1];
            fq[i] = fq[i - 1];
            a0q[i] = a0q[i - 1];
        }
#pragma unroll
        for (int i = 6; i > 0; i--) a2q[i] = a2q[i - 1];
#pragma unroll
        for (int i = 4; i > 0; i--) w[i] = w[i - 1];
        a1q[2] = a1q[1];
        a1q[1] = a1q[0];
        cq[2][0] = ok ? cq[2][0] : 1.0f;
        cq[2][1] = ok ? cq[2][1] : 1.0f;
        // publish plane P
        M.a1[m][0][ty][q] = a1q[2][0];
        M.a1[m][1][ty][q] = a1q[2][1];
        if (!ZERO_IN) M.v[m & 1][ty][q] = w[3];
        __builtin_amdgcn_sched_barrier(0);
        // plane P+2, and vin of P+3 (its second colour's column is X)
        const long long oL = oM;
        const unsigned nL = (unsigned)kM < (unsigned)n2 ? bytes : 0;
        cq[0] = at2(c, oN, nN);
        fq[0] = at2(f, oN, nN);
        a0q[0] = at2(a0, oN, nN);
        a1q[0] = at2(a1, oN, nN);
        if (!ZERO_IN) w[0] = at2(vin, oL, nL)[x];
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        constexpr int m1 = (m + 5) % 6, m2 = (m + 4) % 6, m3 = (m + 3) % 6;
        const int tm = ty > 0 ? ty - 1 : 0, tp = ty < PY - 1 ? ty + 1 : PY - 1;
        // one half-step of column X at plane P - d: y neighbours from F, own: the
        // other column's value there, z neighbours zm / zp
        auto half = [&](auto dd, int sl, const float (*F)[PX / 2], float own, float zm, float zp) -> float {
            constexpr int d = decltype(dd)::value;
            const float ym = F[tm][q], yp = F[tp][q], b1 = M.a1[sl][x][ty][q], b1p = M.a1[sl][x][tp][q];
            const float a0y = a0q[2 + d][y];
            const float xm = x == 0 ? lane_down(own) : own, xp = x == 0 ? own : lane_up(own);
            const float a0p = x == 0 ? a0y : lane_up(a0y);
            float sum = fq[2 + d][x];
            sum = fma_t(-a0q[2 + d][x], xm, sum);
            sum = fma_t(-a0p, xp, sum);
            sum = fma_t(-b1, ym, sum);
            sum = fma_t(-b1p, yp, sum);
            sum = fma_t(-a2q[3 + d][x], zm, sum);
            sum = fma_t(-a2q[2 + d][x], zp, sum);
            return sum / cq[2 + d][x];
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        const float u1 = ZERO_IN ? fq[2][x] / cq[2][x] : half(I0(), m, M.v[m & 1], w[3], w[4], w[2]);
        const float u2 = half(I1(), m1, M.h[0][m1 & 1], h1[0], h1[1], u1);
        const float u3 = half(I2(), m2, M.h[1][m1 & 1], h2[0], h2[1], u2);
        const float u4 = half(I3(), m3, M.h[2][m1 & 1], h3[0], h3[1], u3);
        // read at the next step, after its barrier
        M.h[0][m & 1][ty][q] = u1;
        M.h[1][m & 1][ty][q] = u2;
        M.h[2][m & 1][ty][q] = u3;
        // plane P - 3: h4 on X, h3 (of the last step) on Y; dropped outside the core
        // and the chunk's planes
        {
            f32x2 o;
            o[0] = x == 0 ? u4 : h3[0];
            o[1] = x == 0 ? h3[0] : u4;
            const int s = P - 3;
            const bool sin = s >= k0 && s < k1;
            __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(vout + (sin ? s : 0) * plane), 0,
                                                                         sin ? (int)bytes : 0, 0x00027000);
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, o), r, (int)oS, 0, 0);
        }
        h1[1] = h1[0];
        h1[0] = u1;
        h2[1] = h2[0];
        h2[0] = u2;
        h3[1] = h3[0];
        h3[0] = u3;
        // a2 of P+3 after the last use of P-3's, so that its registers are free
        __builtin_amdgcn_sched_barrier(0);
        a2q[0] = at2(a2, oL, nL);
        __builtin_amdgcn_sched_barrier(0);
        oN = oL;
        nN = nL;
        const bool wrap = per2 && kM + 1 == n2;
        kM = wrap ? 0 : kM + 1;
        oM = wrap ? 0 : oM + plane;
        P++;
    };
    // six steps: the period of the queues' registers and of the LDS slots
    while (P - 3 < k1) {
        step(std::integral_constant<int, 0>());
        step(std::integral_constant<int, 1>());
        step(std::integral_constant<int, 2>());
        step(std::integral_constant<int, 3>());
        step(std::integral_constant<int, 4>());
        step(std::integral_constant<int, 5>());
    }
}

template <bool ZERO_IN>
__global__ void __launch_bounds__(1024) k_sweep2_pair(Geo g, const float *__restrict__ c, const float *__restrict__ a0,
                                                      const float *__restrict__ a1, const float *__restrict__ a2,
                                                      const float *__restrict__ f, const float *__restrict__ vin,
                                                      float *__restrict__ vout, int c1, int kc, int gx, int gy) {
    __shared__ PairLds M;
    int bx, by, bz;
    tile_of(gx, gy, bx, by, bz);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane & 31, ty = wv + 16 * (lane >> 5);
    const int iu = bx * (PX - 2 * PR) - PR + 2 * q, ju = by * (PY - 2 * PR) - PR + ty;
    const int ii = wrapc(iu, g.n0, g.p0), jj = wrapc(ju, g.n1, g.p1);
    const bool valid = ii >= 0 && jj >= 0;
    const unsigned oE = valid ? 4u * (unsigned)(jj * g.n0 + ii) : 0xFFFFFFF8u;
    const bool core = 2 * q >= PR && 2 * q < PX - PR && ty >= PR && ty < PY - PR && iu < g.n0 && ju < g.n1;
    const unsigned oS = core ? oE : 0xFFFFFFF8u;
    const int k0 = bz * kc, k1 = min(g.n2, k0 + kc);
    // colour (x + j + k) & 1 of the cell that is A at the first plane, k0 - 3
    const int S = (c1 + by * (PY - 2 * PR) - PR + wv + k0 - 3) & 1;
    if (S == 0)
        pair_march<ZERO_IN, 0>(M, g, c, a0, a1, a2, f, vin, vout, k0, k1, ty, q, valid, oE, oS);
    else
        pair_march<ZERO_IN, 1>(M, g, c, a0, a1, a2, f, vin, vout, k0, k1, ty, q, valid, oE, oS);
}

// ------------------------------------------------------------------ restriction
__device__ __forceinline__ int gdim_(const Geo &g, int d) { return d == 0 ? g.n0 : (d == 1 ? g.n1 : g.n2); }
__device__ __forceinline__ int gper_(const Geo &g, int d) { return d == 0 ? g.p0 : (d == 1 ? g.p1 : g.p2); }

// vout = vin + P vc: one thread per fine cell (vout may alias vin)
template <typename T, int D>
__global__ void __launch_bounds__(256) k_prolong_t(Geo F, Geo C, const T *__restrict__ pm, const T *__restrict__ pp,
                                                   const T *__restrict__ vc, const T *vin, T *vout) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= F.n0 || j >= F.n1) return;
    const int p = (k * F.n1 + j) * F.n0 + i;
    const int fd = D == 0 ? i : (D == 1 ? j : k);
    const int Jd = fd >> 1;
    const int I = D == 0 ? Jd : i, J = D == 1 ? Jd : j, K = D == 2 ? Jd : k;
    const int pl = (K * C.n1 + J) * C.n0 + I;
    T add;
    if ((fd & 1) == 0) {
        add = vc[pl];
    } else {
        add = pm[pl] * vc[pl];
        const int nc = D == 0 ? C.n0 : (D == 1 ? C.n1 : C.n2);
        const int cper = D == 0 ? C.p0 : (D == 1 ? C.p1 : C.p2);
        const int jr = nbp(Jd, nc, cper);
        if (jr >= 0) {
            const int pr = D == 0 ? (K * C.n1 + J) * C.n0 + jr : (D == 1 ? (K * C.n1 + jr) * C.n0 + I
                                                                          : (jr * C.n1 + J) * C.n0 + I);
            add = fma_t(pp[pl], vc[pr], add);
        }
    }
    vout[p] = (vin ? vin[p] : T(0)) + add;
}

// The same prolongation for coarsening in y (D = 1) or z (D = 2) on levels
// whose x rows hold a multiple of CPL cells: CPL consecutive fine cells per
// thread, 16-byte accesses, per cell the arithmetic of k_prolong_t.
template <typename T, int CPL, int D>
__global__ void __launch_bounds__(256) k_prolong_v(Geo F, Geo C, const T *__restrict__ pm, const T *__restrict__ pp,
                                                   const T *__restrict__ vc, const T *vin, T *vout) {
#pragma clang fp contract(off)
    static_assert(D == 1 || D == 2, "x coarsening has no vector form");
    typedef Vec<T, CPL> V;
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) * CPL;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i >= F.n0 || j >= F.n1) return;
    const int p = (k * F.n1 + j) * F.n0 + i;
    const int fd = D == 1 ? j : k;
    const int Jd = fd >> 1;
    const int J = D == 1 ? Jd : j, K = D == 2 ? Jd : k;
    const int pl = (K * C.n1 + J) * C.n0 + i;
    V add;
    if ((fd & 1) == 0) {
        add = vld<T, CPL>(vc + pl);
    } else {
        const V w = vld<T, CPL>(pm + pl), x = vld<T, CPL>(vc + pl);
#pragma unroll
        for (int q = 0; q < CPL; q++) add.v[q] = w.v[q] * x.v[q];
        const int jr = nbp(Jd, D == 1 ? C.n1 : C.n2, D == 1 ? C.p1 : C.p2);
        if (jr >= 0) {
            const int pr = D == 1 ? (K * C.n1 + jr) * C.n0 + i : (jr * C.n1 + J) * C.n0 + i;
            const V w2 = vld<T, CPL>(pp + pl), x2 = vld<T, CPL>(vc + pr);
#pragma unroll
            for (int q = 0; q < CPL; q++) add.v[q] = fma_t(w2.v[q], x2.v[q], add.v[q]);
        }
    }
    // vin may be vout: this thread reads its cells before it writes them
    V a;
    if (vin) {
        a = *reinterpret_cast<const V *>(vin + p);
    } else {
#pragma unroll
        for (int q = 0; q < CPL; q++) a.v[q] = T(0);
    }
    V o;
#pragma unroll
    for (int q = 0; q < CPL; q++) o.v[q] = a.v[q] + add.v[q];
    *reinterpret_cast<V *>(vout + p) = o;
}

// The prolongation for coarsening in x on levels whose rows hold a multiple
// of 2 CPL fine cells: CPL fine cells per thread (16-byte accesses to vin and
// vout), over CPL / 2 coarse cells and the next one to the right. Per cell
// the arithmetic of k_prolong_t<T, 0>.
template <typename T, int CPL>
__global__ void __launch_bounds__(256) k_prolong_xv(Geo F, Geo C, const T *__restrict__ pm, const T *__restrict__ pp,
                                                    const T *__restrict__ vc, const T *vin, T *vout) {
#pragma clang fp contract(off)
    typedef Vec<T, CPL> V;
    constexpr int H = CPL / 2;
    const int i0 = (blockIdx.x * blockDim.x + threadIdx.x) * CPL;
    const int j = blockIdx.y * blockDim.y + threadIdx.y;
    const int k = blockIdx.z;
    if (i0 >= F.n0 || j >= F.n1) return;
    const int rowc = (k * C.n1 + j) * C.n0, p = (k * F.n1 + j) * F.n0 + i0;
    const int J0 = i0 >> 1;
    T cv[H + 1], cm[H], cp[H];
#pragma unroll
    for (int q = 0; q < H; q++) {
        cv[q] = vc[rowc + J0 + q];
        cm[q] = pm[rowc + J0 + q];
        cp[q] = pp[rowc + J0 + q];
    }
    const int jr = nbp(J0 + H - 1, C.n0, C.p0);
    cv[H] = jr >= 0 ? vc[rowc + jr] : T(0);
    V a;  // vin may be vout: read before the write below
    if (vin) {
        a = *reinterpret_cast<const V *>(vin + p);
    } else {
#pragma unroll
        for (int q = 0; q < CPL; q++) a.v[q] = T(0);
    }
    V o;
#pragma unroll
    for (int q = 0; q < CPL; q++) {
        const int h = q >> 1;
        T add;
        if ((q & 1) == 0) {
            add = cv[h];
        } else {
            add = cm[h] * cv[h];
            // the right neighbour exists for every coarse cell but a wall-side last one
            if (h < H - 1 || jr >= 0) add = fma_t(cp[h], cv[h + 1], add);
        }
        o.v[q] = a.v[q] + add;
    }
    *reinterpret_cast<V *>(vout + p) = o;
}

// coarsest level: v = Ainv f, one wavefront per row (Ainv symmetric)
template <typename Tin, typename Tout>
__global__ void __launch_bounds__(256) k_dense_t(int n, const double *__restrict__ Ainv, const Tin *__restrict__ f,
                                                 Tout *__restrict__ v) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= n) return;
    double s = 0.0;
    for (int j = lane; j < n; j += 64) s += Ainv[(long long)row * n + j] * (double)f[j];
    s = wave_sum(s);
    if (lane == 0) v[row] = (Tout)s;
}

// ------------------------------------------------------------------ bottom of the V-cycle
// The small levels (bottom_fits() below), from the pre-smoothing of the first
// of them through the dense coarsest solve back to its post-smoothing, in one
// workgroup of 1024 threads with a barrier between phases. On these levels
// every launch of the per-level kernels costs a few microseconds of latency for
// a few thousand cells of work. Every sum keeps the order and the roundings of
// the per-level kernels of short rows, and sweeps in place equal the out-of-place
// ones (each colour reads only the other colour), so the results are theirs bit
// for bit (rows of 64 FP64 or 128 FP32 cells and more: but for the rounding of
// the residual's first two products, see bottom_fits).
//
// A phase is bound by latency: its loads, the chain of six multiply-adds, the
// division, the barrier. So everything is in LDS: at the start the coefficients
// of all levels are copied there with all loads in flight, and the right-hand
// sides and iterates of the way down stay there for the way up. A thread owns
// one cell of either colour of a level and holds its coefficients, right-hand
// side and neighbour places in registers through the level's phases. The
// iterate in work is stored by colour: with h = ceil(n0 / 2) cells of a colour
// per row and H = h n1 n2, cell (x, j, k) of colour c = (x + j + k) & 1 lies at
// c H + (k n1 + j) h + x / 2: all neighbours are of the other colour, each
// phase reads one half with unit stride, and no lane idles on the other
// colour's cells.
// Beyond the latency a level costs its instructions (16 waves on one CU: 16
// cycles each), so red and black cell share one set of indices, waves without
// cells wait at the barriers, and the code is kept small (a workgroup passes
// through it once: versions with several cells per thread for levels up to 8192
// cells spent 150 us and more fetching instructions).
// FP32 V(2,2), the levels of 1024 cells and below of the 256^3 channel: 56 us
// with indices and global loads in every phase; 35 us now with the level of 2048
// cells too, which took 29 us in nine launches. FP64 V(1,1), 64^3 periodic: 29
// against 22 us.
namespace {

constexpr int BT_THREADS = 1024;
constexpr int BT_LDS = 158 * 1024;  // bytes of LDS the kernel uses

// q = p / d for 0 <= p < 2^24 from a float reciprocal, corrected to exact
__device__ __forceinline__ int bt_div(int p, int d, float inv) {
    int q = (int)((float)p * inv);
    if (q * d > p) q--;
    if ((q + 1) * d <= p) q++;
    return q;
}

// place of a cell in a level's colour-split iterate, h = ceil(n0 / 2), H = h n1 n2
__device__ __forceinline__ int bt_at(const Geo &g, int h, int H, int x, int j, int k) {
    return ((x + j + k) & 1) * H + (k * g.n1 + j) * h + (x >> 1);
}

// One cell of a thread: diagonal, right-hand side, the couplings to its six
// neighbours (0 where there is none), their places in the other colour's half,
// its own place, its x and its flat index (-1: no cell)
template <typename T>
struct BtCell {
    T c, f, a[6];
    int nb[6];
    int at, x, p;
};

// A thread's red and black cell of a level: x = 2 u and 2 u + 1 of row (j, k)
template <typename T>
struct BtPair {
    BtCell<T> r, b;
    int j, k;
};

// q = the place in a colour (q < H), A = c, a0, a1, a2 (N entries each)
template <typename T>
__device__ __forceinline__ void bt_pair(const Geo &g, float ih, float i1, int q, const T *A, BtPair<T> &S) {
    const int h = (g.n0 + 1) >> 1, H = h * g.n1 * g.n2, N = (int)g.N, plane = g.n0 * g.n1;
    const int row = bt_div(q, h, ih), u = q - row * h;
    const int k = bt_div(row, g.n1, i1), j = row - k * g.n1;
    const int e = (j + k) & 1;  // colour of the even cell
    const bool odd = 2 * u + 1 < g.n0;
    const int p0 = row * g.n0 + 2 * u, p1 = odd ? p0 + 1 : p0;  // a missing odd cell loads the even one's
    const T *a0 = A + N, *a1 = A + 2 * N, *a2 = A + 3 * N;
    // x: even - left uL, right u; odd - left u, right uR (place in the row, -1: none)
    const int uL = u > 0 ? u - 1 : (g.p0 ? h - 1 : -1);
    const int uR = 2 * u + 2 < g.n0 ? u + 1 : (g.p0 && g.n0 > 1 ? 0 : -1);
    const int q0 = row * h;
    // y, z: the same place of the neighbouring rows; a direction of one cell has
    // no neighbour (a periodic one couples to itself with 0)
    const int jm = j > 0 ? -1 : (g.p1 ? g.n1 - 1 : 0), jp = j < g.n1 - 1 ? 1 : (g.p1 ? 1 - g.n1 : 0);
    const int km = k > 0 ? -1 : (g.p2 ? g.n2 - 1 : 0), kp = k < g.n2 - 1 ? 1 : (g.p2 ? 1 - g.n2 : 0);
    const int hn = h * g.n1;
    const int qym = q + jm * h, qyp = q + jp * h, qzm = q + km * hn, qzp = q + kp * hn;
    const T z = T(0);
    const T cE = A[p0], cO = A[p1];
    const T xE = a0[p0], xO = a0[p1], xN = a0[row * g.n0 + (uR >= 0 ? 2 * uR : 0)];
    const T ymE = a1[p0], ymO = a1[p1], ypE = a1[p0 + jp * g.n0], ypO = a1[p1 + jp * g.n0];
    const T zmE = a2[p0], zmO = a2[p1], zpE = a2[p0 + kp * plane], zpO = a2[p1 + kp * plane];
    auto fill = [=](BtCell<T> &C, int col, bool even) {
        const int o = (col ^ 1) * H;
        const bool hl = even ? uL >= 0 : true, hr = even ? odd : uR >= 0;
        C.c = even ? cE : cO;
        C.a[0] = hl ? (even ? xE : xO) : z;
        C.a[1] = hr ? (even ? xO : xN) : z;
        C.a[2] = jm ? (even ? ymE : ymO) : z;
        C.a[3] = jp ? (even ? ypE : ypO) : z;
        C.a[4] = km ? (even ? zmE : zmO) : z;
        C.a[5] = kp ? (even ? zpE : zpO) : z;
        C.nb[0] = o + q0 + (hl ? (even ? uL : u) : u);
        C.nb[1] = o + q0 + (hr ? (even ? u : uR) : u);
        C.nb[2] = o + qym;
        C.nb[3] = o + qyp;
        C.nb[4] = o + qzm;
        C.nb[5] = o + qzp;
        C.at = col * H + q;
        C.x = 2 * u + (even ? 0 : 1);
        C.p = even ? p0 : (odd ? p1 : -1);
    };
    fill(S.r, 0, e == 0);
    fill(S.b, 1, e == 1);
    S.j = j;
    S.k = k;
}

// (f - sum a v_nb) / c in the order and with the roundings of the per-level
// sweeps: each multiply-add rounds once, explicitly, as the conditional ones
// there do (a plain c v + a v' may be fused either way)
template <typename T>
__device__ __forceinline__ void bt_relax(const BtCell<T> &S, T *V) {
#pragma clang fp contract(off)
    T v[6];
#pragma unroll
    for (int d = 0; d < 6; d++) v[d] = V[S.nb[d]];
    T sum = S.f;
#pragma unroll
    for (int d = 0; d < 6; d++) sum = fma_t(-S.a[d], v[d], sum);
    if (S.p >= 0) V[S.at] = sum / S.c;
}

// R[p] = f - A v, and the iterate to K[p]
template <typename T>
__device__ __forceinline__ void bt_resid(const BtCell<T> &S, const T *V, T *R, T *K) {
#pragma clang fp contract(off)
    if (S.p < 0) return;
    const T vc = V[S.at];
    T t = S.c * vc;
#pragma unroll
    for (int d = 0; d < 6; d++) t = fma_t(S.a[d], V[S.nb[d]], t);
    R[S.p] = S.f - t;
    K[S.p] = vc;
}

// (P^T r) at coarse cell (I, J, K) along direction d (as k_gather_t), r by flat index
template <typename T>
__device__ __forceinline__ T bt_gather(const Geo &F, const Geo &C, const BotDir &D, const T *R, const T *pm,
                                       const T *pp, int I, int J, int K) {
#pragma clang fp contract(off)
    const int d = D.d, nd = D.nf, per = D.per, nc = D.nc, sf = D.sf, sc = D.sc;
    const int Jd = d == 0 ? I : (d == 1 ? J : K);
    const int pc = (K * C.n1 + J) * C.n0 + I;
    const int pf = ((d == 2 ? 2 * K : K) * F.n1 + (d == 1 ? 2 * J : J)) * F.n0 + (d == 0 ? 2 * I : I);
    const bool hasl = Jd > 0 || per, hasr = 2 * Jd + 1 < nd;
    const int pl = Jd > 0 ? pf - sf : (per ? pf + (nd - 1) * sf : pf);
    const int wl = Jd > 0 ? pc - sc : (per ? pc + (nc - 1) * sc : pc);
    const T wm = pm[pc], wp = pp[wl], rr = R[hasr ? pf + sf : pf], rl = R[pl];
    T s = R[pf];
    if (hasr) s = fma_t(wm, rr, s);
    if (hasl) s = fma_t(wp, rl, s);
    return s;
}

// (P vc) at fine cell (i, j, k) along direction d (as k_prolong_t), vc stored by colour
template <typename T>
__device__ __forceinline__ T bt_prolong(const Geo &C, const BotDir &D, const T *pm, const T *pp, const T *vc, int i,
                                        int j, int k) {
#pragma clang fp contract(off)
    const int h = (C.n0 + 1) >> 1, H = h * C.n1 * C.n2, d = D.d, nc = D.nc, per = D.per;
    const int fd = d == 0 ? i : (d == 1 ? j : k), Jd = fd >> 1;
    const int I = d == 0 ? Jd : i, J = d == 1 ? Jd : j, K = d == 2 ? Jd : k;
    const bool hasr = Jd < nc - 1 || per;
    const int jr = Jd < nc - 1 ? Jd + 1 : (per ? 0 : Jd);
    const int pl = (K * C.n1 + J) * C.n0 + I;
    const T x0 = vc[bt_at(C, h, H, I, J, K)];
    const T x1 = vc[bt_at(C, h, H, d == 0 ? jr : I, d == 1 ? jr : J, d == 2 ? jr : K)];
    const T m = pm[pl] * x0, q = fma_t(pp[pl], x1, m);
    return (fd & 1) ? (hasr ? q : m) : x0;
}

template <typename T>
__global__ void __launch_bounds__(BT_THREADS) k_bottom(BotArgs<T> a) {
    constexpr int E = BT_LDS / (int)sizeof(T);
    __shared__ T M[E];
    const int nl = a.nlev, npre = a.npre, npost = a.npost, cap = a.cap, tid = (int)threadIdx.x;
    // two iterates by colour and the residual (cap entries each), then per level
    // c, a0, a1, a2, pm, pp, f and the iterate of the way down (N entries each)
    T *R = M + 2 * cap;
#pragma unroll 1
    for (int l = 0, base = 3 * cap; l < nl; l++) {
        const int N = (int)a.L[l].g.N;
        T *d = M + base;
        const T *s0 = a.L[l].c, *s1 = a.L[l].a0, *s2 = a.L[l].a1, *s3 = a.L[l].a2, *s4 = a.L[l].pm, *s5 = a.L[l].pp;
        for (int q = tid; q < N; q += BT_THREADS) {
            const T v0 = s0[q], v1 = s1[q], v2 = s2[q], v3 = s3[q], v4 = s4[q], v5 = s5[q];
            d[q] = v0;
            d[N + q] = v1;
            d[2 * N + q] = v2;
            d[3 * N + q] = v3;
            d[4 * N + q] = v4;
            d[5 * N + q] = v5;
            if (l == 0) d[6 * N + q] = a.L[0].f[q];
        }
        base += 8 * N;
    }
    __syncthreads();
    BtPair<T> S;  // this thread's cells
    // down: pre-smoothing, residual, restriction
    int base = 3 * cap;
#pragma unroll 1
    for (int l = 0; l < nl - 1; l++) {
        const Geo g = a.L[l].g;
        const int N = (int)g.N, relax = a.L[l].relax, H = ((g.n0 + 1) >> 1) * g.n1 * g.n2;
        const bool act = tid < H;
        T *D = M + base, *fs = D + 6 * N;
        if (act) {
            bt_pair<T>(g, a.L[l].ih, a.L[l].i1, tid, D, S);
            if (l > 0) {
                const Geo F = a.L[l - 1].g;
                const BotDir d = a.L[l - 1].dir;
                if (S.r.p >= 0) fs[S.r.p] = bt_gather<T>(F, g, d, R, D + 4 * N, D + 5 * N, S.r.x, S.j, S.k);
                if (S.b.p >= 0) fs[S.b.p] = bt_gather<T>(F, g, d, R, D + 4 * N, D + 5 * N, S.b.x, S.j, S.k);
            }
            S.r.f = fs[S.r.p >= 0 ? S.r.p : 0];
            S.b.f = fs[S.b.p >= 0 ? S.b.p : 0];
        }
        if (!relax) {
            // skipped level: v = 0 (the prolongation adds to it), f restricted as it is
            __syncthreads();  // R has been read
            if (act) {
                if (S.r.p >= 0) R[S.r.p] = S.r.f;
                if (S.b.p >= 0) R[S.b.p] = S.b.f;
            }
        } else {
            // the first colour from zero; places without a cell are read with a zero coupling
            if (act) {
                M[S.r.at] = S.r.p >= 0 ? S.r.f / S.r.c : T(0);
                M[S.b.at] = T(0);
            }
#pragma unroll 1
            for (int sw = 0;;) {
                __syncthreads();
                if (act) bt_relax<T>(S.b, M);
                __syncthreads();
                if (++sw == npre) break;
                if (act) bt_relax<T>(S.r, M);
            }
            if (act) {
                bt_resid<T>(S.r, M, R, D + 7 * N);
                bt_resid<T>(S.b, M, R, D + 7 * N);
            }
        }
        __syncthreads();
        base += 8 * N;
    }
    // coarsest: v = Ainv f, one wavefront per row (lane-strided columns, as k_dense_t)
    {
        const Geo C = a.L[nl - 1].g, F = a.L[nl - 2].g;
        const BotDir d = a.L[nl - 2].dir;
        const int n = (int)C.N, h = (C.n0 + 1) >> 1, H = h * C.n1 * C.n2;
        const double *Ainv = a.Ainv;
        T *D = M + base, *fc = D + 6 * n, *vc = D + 7 * n;
        int i = 0, j = 0, k = 0;
        if (tid < n) {
            const int r = bt_div(tid, C.n0, 1.0f / (float)C.n0);
            i = tid - r * C.n0;
            k = bt_div(r, C.n1, a.L[nl - 1].i1);
            j = r - k * C.n1;
            fc[tid] = bt_gather<T>(F, C, d, R, D + 4 * n, D + 5 * n, i, j, k);
        }
        __syncthreads();
        const int lane = tid & 63, wave = tid >> 6;
#pragma unroll 4
        for (int row = wave; row < n; row += BT_THREADS / 64) {
            double s = 0.0;
            for (int jj = lane; jj < n; jj += 64) s += Ainv[(long long)row * n + jj] * (double)fc[jj];
            s = wave_sum(s);
            if (lane == 0) vc[row] = (T)s;
        }
        __syncthreads();
        if (tid < n) M[bt_at(C, h, H, i, j, k)] = vc[tid];
        __syncthreads();
    }
    // up: prolongation and post-smoothing (the other colour first)
    int vb = 0;
#pragma unroll 1
    for (int l = nl - 2; l >= 0; l--) {
        const Geo g = a.L[l].g, C = a.L[l + 1].g;
        const int N = (int)g.N, NC = (int)C.N, relax = a.L[l].relax;
        const BotDir d = a.L[l].dir;
        const bool act = tid < ((g.n0 + 1) >> 1) * g.n1 * g.n2;
        const T *pm = M + base + 4 * NC, *pp = M + base + 5 * NC, *vc = M + vb * cap;
        base -= 8 * N;
        const T *D = M + base;
        vb ^= 1;
        T *V = M + vb * cap;
        if (act) {
            bt_pair<T>(g, a.L[l].ih, a.L[l].i1, tid, D, S);
            const int rp = S.r.p >= 0 ? S.r.p : 0, bp = S.b.p >= 0 ? S.b.p : 0;
            S.r.f = D[6 * N + rp];
            S.b.f = D[6 * N + bp];
            // a missing cell's x is the last one's here
            const int rx = S.r.p >= 0 ? S.r.x : S.b.x, bx = S.b.p >= 0 ? S.b.x : S.r.x;
            const T rv = (relax ? D[7 * N + rp] : T(0)) + bt_prolong<T>(C, d, pm, pp, vc, rx, S.j, S.k);
            const T bv = (relax ? D[7 * N + bp] : T(0)) + bt_prolong<T>(C, d, pm, pp, vc, bx, S.j, S.k);
            V[S.r.at] = S.r.p >= 0 ? rv : T(0);
            V[S.b.at] = S.b.p >= 0 ? bv : T(0);
        }
        __syncthreads();
        if (relax)
#pragma unroll 1
            for (int sw = 0; sw < npost; sw++) {
                if (act) bt_relax<T>(S.b, V);
                __syncthreads();
                if (act) bt_relax<T>(S.r, V);
                __syncthreads();
            }
        if (l == 0 && act) {
            T *vout = a.L[0].v;
            if (S.r.p >= 0) vout[S.r.p] = V[S.r.at];
            if (S.b.p >= 0) vout[S.b.p] = V[S.b.at];
        }
    }
}

}  // namespace

// levels whose rows are long enough for the row-wave kernels (k_stencil_rw)
template <typename T>
static bool row_waves(const Geo &g) {
    constexpr int CPL = 16 / sizeof(T);
    return g.n0 % CPL == 0 && g.n0 >= 32 * CPL;
}

// Whether levels of these shapes, first to coarsest, are the bottom kernel's:
// one cell of a colour per thread, and all arrays in its LDS (2048 FP32 or 1024
// FP64 cells in the first level of a halving sequence). Beyond 1024 cells, levels
// with rows long enough for k_stencil_rw stay out: that kernel's residual fuses the
// first two products the other way round, so the cycle's bits would change.
static long long bottom_places(const Geo &g) { return 2LL * ((g.n0 + 1) / 2) * g.n1 * g.n2; }

template <typename T>
bool bottom_fits(const Geo *g, int n) {
    long long cap = 0, cells = 0;
    for (int l = 0; l < n; l++) {
        const long long q = bottom_places(g[l]);
        if (l < n - 1 && (q > 2 * BT_THREADS || (g[l].N > 1024 && row_waves<T>(g[l])))) return false;
        cap = std::max(cap, q);
        cells += g[l].N;
    }
    return (3 * cap + 8 * cells) * (long long)sizeof(T) <= BT_LDS;
}

template <typename T>
void launch_bottom(hipStream_t s, const BotArgs<T> &args) {
    BotArgs<T> a = args;
    long long cap = 0;
    for (int l = 0; l < a.nlev; l++) {
        const Geo &g = a.L[l].g;
        cap = std::max(cap, bottom_places(g));
        a.L[l].ih = 1.0f / (float)((g.n0 + 1) / 2);
        a.L[l].i1 = 1.0f / (float)g.n1;
        if (l + 1 < a.nlev) {
            const Geo &c = a.L[l + 1].g;
            BotDir &D = a.L[l].dir;
            const int nf[3] = {g.n0, g.n1, g.n2}, nc[3] = {c.n0, c.n1, c.n2}, per[3] = {g.p0, g.p1, g.p2};
            D.nf = nf[D.d];
            D.nc = nc[D.d];
            D.per = per[D.d];
            D.sf = D.d == 0 ? 1 : (D.d == 1 ? g.n0 : g.n0 * g.n1);
            D.sc = D.d == 0 ? 1 : (D.d == 1 ? c.n0 : c.n0 * c.n1);
        }
    }
    a.cap = (int)cap;
    hipLaunchKernelGGL(k_bottom<T>, dim3(1), dim3(BT_THREADS), 0, s, a);
}

// ------------------------------------------------------------------ launchers

namespace {
int pow2ceil(int v) {
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}
}  // namespace

// x-y tile for 256-thread blocks adapted to small planes
void tile_dims(const Geo &g, int &tx, int &ty) {
    tx = std::min(64, pow2ceil(g.n0));
    ty = std::min(256 / tx, pow2ceil(g.n1));
}

// 256-thread blocks for the vector transfers: x threads own cpl cells each
static void vec_tile_dims(const Geo &g, int cpl, int &tx, int &ty) {
    tx = std::min(64, pow2ceil(g.n0 / cpl));
    ty = std::min(256 / tx, pow2ceil(g.n1));
}

static bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// z chunk for the tiled march kernels (256-thread blocks)
int march_blocks(const Geo &g, int &kc) {
    int tx, ty;
    tile_dims(g, tx, ty);
    const int gx = (g.n0 + tx - 1) / tx, gy = (g.n1 + ty - 1) / ty;
    long long tiles = (long long)gx * gy;
    long long want = 4096;  // 256-thread blocks; z chunks of ~16 planes at 256^3
    kc = (int)std::max<long long>(1, (g.n2 * tiles + want - 1) / want);
    if (kc > g.n2) kc = g.n2;
    int gz = (g.n2 + kc - 1) / kc;
    while ((long long)gz * tiles > MAX_PARTS && kc < g.n2) {
        kc++;
        gz = (g.n2 + kc - 1) / kc;
    }
    return (int)(tiles * gz);
}

// launch shape of the SpMV: row waves (CPL cells of T per lane, 16 B) when
// the rows are long enough and a multiple of CPL, else the tiled march
struct ApplyCfg {
    bool rw;
    int kc, gx, gy, gz;
    int blocks;
};

template <typename T>
ApplyCfg apply_cfg(const Geo &g) {
    constexpr int CPL = 16 / sizeof(T);
    ApplyCfg a{};
    if (row_waves<T>(g)) {
        a.rw = true;
        a.gx = (g.n0 + 64 * CPL - 1) / (64 * CPL);
        a.gy = (g.n1 + 3) / 4;
        const long long tiles = (long long)a.gx * a.gy;
        // z chunks of ~4 planes at 256^3 (measured best among 4, 8, 16 for both
        // precisions: 5.6 TB/s FP32, 5.1 TB/s FP64 in a standalone SpMV)
        const long long want = 1024 * (long long)sizeof(T);
        a.kc = (int)std::max<long long>(1, (g.n2 * tiles + want - 1) / want);
        if (a.kc > g.n2) a.kc = g.n2;
        a.gz = (g.n2 + a.kc - 1) / a.kc;
        while ((long long)a.gz * tiles > MAX_PARTS && a.kc < g.n2) {
            a.kc++;
            a.gz = (g.n2 + a.kc - 1) / a.kc;
        }
        a.blocks = (int)(tiles * a.gz);
        return a;
    }
    a.rw = false;
    int tx, ty;
    tile_dims(g, tx, ty);
    a.blocks = march_blocks(g, a.kc);
    a.gx = (g.n0 + tx - 1) / tx;
    a.gy = (g.n1 + ty - 1) / ty;
    a.gz = (g.n2 + a.kc - 1) / a.kc;
    return a;
}

// workgroups of the FP64 SpMV (one partial of <x, Ax> each)
int apply_blocks(const Geo &g, int &kc) {
    const ApplyCfg a = apply_cfg<double>(g);
    kc = a.kc;
    return a.blocks;
}

template <typename T>
void launch_apply(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *x, T *y,
                  double *part) {
    const ApplyCfg a = apply_cfg<T>(g);
    if (a.rw) {
        hipLaunchKernelGGL((k_stencil_rw<T, 16 / sizeof(T), RW_APPLY>), dim3(a.blocks), dim3(256), 0, s, g, c, a0, a1,
                           a2, (const T *)nullptr, x, y, part, 0, a.kc, a.gx, a.gy);
        return;
    }
    int tx, ty;
    tile_dims(g, tx, ty);
    hipLaunchKernelGGL(k_apply_t<T>, dim3(a.blocks), dim3(tx, ty), 0, s, g, c, a0, a1, a2, x, y, part, a.kc, a.gx,
                       a.gy);
}

void launch_apply_x32(hipStream_t s, const Geo &g, const double *c, const double *a0, const double *a1,
                      const double *a2, const float *x, double *y, double *part) {
    const ApplyCfg a = apply_cfg<double>(g);
    if (a.rw) {
        hipLaunchKernelGGL((k_stencil_rw<double, 2, RW_APPLY, float>), dim3(a.blocks), dim3(256), 0, s, g, c, a0, a1,
                           a2, (const double *)nullptr, x, y, part, 0, a.kc, a.gx, a.gy);
        return;
    }
    int tx, ty;
    tile_dims(g, tx, ty);
    hipLaunchKernelGGL((k_apply_t<double, float>), dim3(a.blocks), dim3(tx, ty), 0, s, g, c, a0, a1, a2, x, y, part,
                       a.kc, a.gx, a.gy);
}

template <typename T>
void launch_smooth0(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f, T *v,
                    int c1) {
    const ApplyCfg a = apply_cfg<T>(g);
    if (a.rw) {
        hipLaunchKernelGGL((k_stencil_rw<T, 16 / sizeof(T), RW_SMOOTH0>), dim3(a.blocks), dim3(256), 0, s, g, c, a0,
                           a1, a2, f, (const T *)nullptr, v, (double *)nullptr, c1, a.kc, a.gx, a.gy);
        return;
    }
    int tx, ty, kc;
    tile_dims(g, tx, ty);
    march_blocks(g, kc);
    const int gx = (g.n0 + tx - 1) / tx, gy = (g.n1 + ty - 1) / ty, gz = (g.n2 + kc - 1) / kc;
    hipLaunchKernelGGL(k_smooth0_t<T>, dim3(gx * gy * gz), dim3(tx, ty), 0, s, g, c, a0, a1, a2, f, v, c1, kc, gx,
                       gy);
}

template <typename T>
void launch_resid(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f,
                  const T *x, T *r) {
    const ApplyCfg a = apply_cfg<T>(g);
    if (a.rw) {
        hipLaunchKernelGGL((k_stencil_rw<T, 16 / sizeof(T), RW_RESID>), dim3(a.blocks), dim3(256), 0, s, g, c, a0, a1,
                           a2, f, x, r, (double *)nullptr, 0, a.kc, a.gx, a.gy);
        return;
    }
    int tx, ty, kc;
    tile_dims(g, tx, ty);
    march_blocks(g, kc);
    const int gx = (g.n0 + tx - 1) / tx, gy = (g.n1 + ty - 1) / ty, gz = (g.n2 + kc - 1) / kc;
    hipLaunchKernelGGL(k_resid_t<T>, dim3(gx * gy * gz), dim3(tx, ty), 0, s, g, c, a0, a1, a2, f, x, r, kc, gx,
                       gy);
}

template <typename T>
void launch_gather(hipStream_t s, const Geo &F, const Geo &C, int d, const T *r, const T *pm, const T *pp, T *fc,
                   bool vec) {
    constexpr int CPL = 16 / sizeof(T);
    if (vec && d == 0 && F.n0 % (2 * CPL) == 0 && aligned16(r) && aligned16(pm) && aligned16(pp) && aligned16(fc)) {
        int tx, ty;
        vec_tile_dims(C, CPL, tx, ty);
        dim3 grid((C.n0 / CPL + tx - 1) / tx, (C.n1 + ty - 1) / ty, C.n2);
        hipLaunchKernelGGL((k_gather_xv<T, CPL>), grid, dim3(tx, ty), 0, s, F, C, r, pm, pp, fc);
        return;
    }
    if (vec && d != 0 && F.n0 % CPL == 0 && aligned16(r) && aligned16(pm) && aligned16(pp) && aligned16(fc)) {
        int tx, ty;
        vec_tile_dims(C, CPL, tx, ty);
        dim3 grid((C.n0 / CPL + tx - 1) / tx, (C.n1 + ty - 1) / ty, C.n2);
        if (d == 1)
            hipLaunchKernelGGL((k_gather_v<T, CPL, 1>), grid, dim3(tx, ty), 0, s, F, C, r, pm, pp, fc);
        else
            hipLaunchKernelGGL((k_gather_v<T, CPL, 2>), grid, dim3(tx, ty), 0, s, F, C, r, pm, pp, fc);
        return;
    }
    int tx, ty;
    tile_dims(C, tx, ty);
    dim3 grid((C.n0 + tx - 1) / tx, (C.n1 + ty - 1) / ty, C.n2);
    if (d == 0)
        hipLaunchKernelGGL((k_gather_t<T, 0>), grid, dim3(tx, ty), 0, s, F, C, r, pm, pp, fc);
    else if (d == 1)
        hipLaunchKernelGGL((k_gather_t<T, 1>), grid, dim3(tx, ty), 0, s, F, C, r, pm, pp, fc);
    else
        hipLaunchKernelGGL((k_gather_t<T, 2>), grid, dim3(tx, ty), 0, s, F, C, r, pm, pp, fc);
}

template <typename T, int SY>
static void launch_sweep_sy(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2,
                            const T *f, const T *vin, T *vout, int c1, long long target) {
    const int gx = (g.n0 + SX - 3) / (SX - 2), gy = (g.n1 + SY - 3) / (SY - 2);
    const long long tiles = (long long)gx * gy;
    // about `target` workgroups. Each z chunk recomputes 3 planes, so on large
    // levels (bandwidth-bound) chunks stay >= 16 planes when possible; small
    // levels are latency-bound (one barrier per plane), so there the chunks
    // get as short as the target allows.
    long long gz = std::max<long long>(1, target / tiles);
    if (g.N >= (1 << 22) && gz > 1 && (g.n2 + gz - 1) / gz < 16) gz = std::max<long long>(1, g.n2 / 16);
    if (gz > g.n2) gz = g.n2;
    int kc = (int)((g.n2 + gz - 1) / gz);
    if (kc < 1) kc = 1;
    const int nz = (g.n2 + kc - 1) / kc;
    dim3 grid((unsigned)(gx * gy * nz));
    if (vin)
        hipLaunchKernelGGL((k_sweep<T, false, SY>), grid, dim3(SX, SY), 0, s, g, c, a0, a1, a2, f, vin, vout, c1, kc,
                           gx, gy);
    else
        hipLaunchKernelGGL((k_sweep<T, true, SY>), grid, dim3(SX, SY), 0, s, g, c, a0, a1, a2, f,
                           (const T *)nullptr, vout, c1, kc, gx, gy);
}

// 64 x 16 workgroups (1024 threads, two per CU); ~512 of them per launch at
// 256^3 measured best among 64 x {4, 8, 16} tiles and 512..4096 groups. (A
// row-wave variant with 16-byte loads and 14-row workgroups measured slower:
// 183 against 137 us at 256^3, FP32.)
// Whole-row tiles (k_sweep_row) on levels of rows <= 128 cells: about
// `target` workgroups, z chunks of >= ROW_MIN_KC planes on large levels. With
// fewer tiles per plane than k_sweep the same workgroup count leaves shorter
// z chunks, hence fewer plane steps per workgroup.
constexpr int ROW_MIN_KC = 8;

template <typename T, int NX>
static void launch_sweep_row(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2,
                             const T *f, const T *vin, T *vout, int c1, long long target) {
    constexpr int NY = 1024 / NX;
    const int gy = (g.n1 + NY - 3) / (NY - 2);
    long long gz = std::max<long long>(1, target / gy);
    if (g.N >= (1 << 22) && gz > 1 && (g.n2 + gz - 1) / gz < ROW_MIN_KC)
        gz = std::max<long long>(1, g.n2 / ROW_MIN_KC);
    if (gz > g.n2) gz = g.n2;
    int kc = (int)((g.n2 + gz - 1) / gz);
    if (kc < 1) kc = 1;
    const int nz = (g.n2 + kc - 1) / kc;
    dim3 grid((unsigned)(gy * nz)), block(NX, NY);
    if (vin)
        hipLaunchKernelGGL((k_sweep_row<T, false, NX>), grid, block, 0, s, g, c, a0, a1, a2, f, vin, vout, c1, kc, gy);
    else
        hipLaunchKernelGGL((k_sweep_row<T, true, NX>), grid, block, 0, s, g, c, a0, a1, a2, f, (const T *)nullptr,
                           vout, c1, kc, gy);
}

template <typename T>
void launch_sweep(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f,
                  const T *vin, T *vout, int c1, bool tiles) {
    if (!tiles && g.n0 <= 32)
        launch_sweep_row<T, 32>(s, g, c, a0, a1, a2, f, vin, vout, c1, 512);
    else if (!tiles && g.n0 <= 64)
        launch_sweep_row<T, 64>(s, g, c, a0, a1, a2, f, vin, vout, c1, 512);
    else if (!tiles && g.n0 <= 128)
        launch_sweep_row<T, 128>(s, g, c, a0, a1, a2, f, vin, vout, c1, 512);
    else
        launch_sweep_sy<T, 16>(s, g, c, a0, a1, a2, f, vin, vout, c1, 512);
}

// Two sweeps of colour order c1 in one launch: k_sweep2_pair where it can run
// (247 -> 145 us at 256^3), else k_sweep2 with 58 x 10 output tiles, about 512
// workgroups and z chunks of >= 16 planes on large levels (each chunk recomputes
// 6 planes). vin and vout must differ; vin == nullptr: the first sweep starts
// from a zero iterate.
template <typename T>
void launch_sweep2(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f,
                   const T *vin, T *vout, int c1, bool one_cell) {
    if constexpr (std::is_same<T, float>::value) {
        // (8-byte accesses; the level's own buffers always are aligned)
        const auto al = reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(a0) |
                        reinterpret_cast<uintptr_t>(a1) | reinterpret_cast<uintptr_t>(a2) |
                        reinterpret_cast<uintptr_t>(f) | reinterpret_cast<uintptr_t>(vin) |
                        reinterpret_cast<uintptr_t>(vout);
        if (!one_cell && pair_form<T>(g) && al % 8 == 0) {
            const int gx = (g.n0 + PX - 2 * PR - 1) / (PX - 2 * PR), gy = (g.n1 + PY - 2 * PR - 1) / (PY - 2 * PR);
            // one workgroup per CU: z chunks so that about 256 run, each of whole
            // rounds of 6 steps and recomputing 6 planes
            const long long gz = std::max<long long>(1, 256 / ((long long)gx * gy));
            const int kc = (int)(((g.n2 + gz - 1) / gz + 5) / 6 * 6);
            const int nz = (g.n2 + kc - 1) / kc;
            if (vin)
                hipLaunchKernelGGL(k_sweep2_pair<false>, dim3((unsigned)(gx * gy * nz)), dim3(1024), 0, s, g, c, a0, a1,
                                   a2, f, vin, vout, c1, kc, gx, gy);
            else
                hipLaunchKernelGGL(k_sweep2_pair<true>, dim3((unsigned)(gx * gy * nz)), dim3(1024), 0, s, g, c, a0, a1,
                                   a2, f, vin, vout, c1, kc, gx, gy);
            return;
        }
    }
    constexpr int SY = 16;
    const int gx = (g.n0 + SX - 2 * R2 - 1) / (SX - 2 * R2), gy = (g.n1 + SY - 2 * R2 - 1) / (SY - 2 * R2);
    const long long tiles = (long long)gx * gy;
    long long gz = std::max<long long>(1, 512 / tiles);
    if (g.N >= (1 << 22) && gz > 1 && (g.n2 + gz - 1) / gz < 16) gz = std::max<long long>(1, g.n2 / 16);
    if (gz > g.n2) gz = g.n2;
    int kc = (int)((g.n2 + gz - 1) / gz);
    if (kc < 1) kc = 1;
    const int nz = (g.n2 + kc - 1) / kc;
    if (vin)
        hipLaunchKernelGGL((k_sweep2<T, SY, false>), dim3((unsigned)(gx * gy * nz)), dim3(SX, SY), 0, s, g, c, a0, a1,
                           a2, f, vin, vout, c1, kc, gx, gy);
    else
        hipLaunchKernelGGL((k_sweep2<T, SY, true>), dim3((unsigned)(gx * gy * nz)), dim3(SX, SY), 0, s, g, c, a0, a1,
                           a2, f, vin, vout, c1, kc, gx, gy);
}

template <typename T>
void launch_prolong_to(hipStream_t s, const Geo &F, const Geo &C, int d, const T *pm, const T *pp, const T *vc,
                       const T *vin, T *vout, bool vec) {
    constexpr int CPL = 16 / sizeof(T);
    if (vec && d == 0 && F.n0 % (2 * CPL) == 0 && aligned16(vin) && aligned16(vout)) {
        int tx, ty;
        vec_tile_dims(F, CPL, tx, ty);
        dim3 grid((F.n0 / CPL + tx - 1) / tx, (F.n1 + ty - 1) / ty, F.n2);
        hipLaunchKernelGGL((k_prolong_xv<T, CPL>), grid, dim3(tx, ty), 0, s, F, C, pm, pp, vc, vin, vout);
        return;
    }
    if (vec && d != 0 && F.n0 % CPL == 0 && aligned16(pm) && aligned16(pp) && aligned16(vc) && aligned16(vin) &&
        aligned16(vout)) {
        int tx, ty;
        vec_tile_dims(F, CPL, tx, ty);
        dim3 grid((F.n0 / CPL + tx - 1) / tx, (F.n1 + ty - 1) / ty, F.n2);
        if (d == 1)
            hipLaunchKernelGGL((k_prolong_v<T, CPL, 1>), grid, dim3(tx, ty), 0, s, F, C, pm, pp, vc, vin, vout);
        else
            hipLaunchKernelGGL((k_prolong_v<T, CPL, 2>), grid, dim3(tx, ty), 0, s, F, C, pm, pp, vc, vin, vout);
        return;
    }
    int tx, ty;
    tile_dims(F, tx, ty);
    dim3 grid((F.n0 + tx - 1) / tx, (F.n1 + ty - 1) / ty, F.n2);
    if (d == 0)
        hipLaunchKernelGGL((k_prolong_t<T, 0>), grid, dim3(tx, ty), 0, s, F, C, pm, pp, vc, vin, vout);
    else if (d == 1)
        hipLaunchKernelGGL((k_prolong_t<T, 1>), grid, dim3(tx, ty), 0, s, F, C, pm, pp, vc, vin, vout);
    else
        hipLaunchKernelGGL((k_prolong_t<T, 2>), grid, dim3(tx, ty), 0, s, F, C, pm, pp, vc, vin, vout);
}

// order: chain_order of the directions
template <typename T, typename F>
static void launch_chain(const Geo *g, int order, const T *const *pm, const T *const *pp, F launch) {
    Chain<T> ch;
    for (int i = 0; i < 4; i++) ch.g[i] = g[i];
    for (int i = 0; i < 3; i++) ch.pm[i] = pm[i], ch.pp[i] = pp[i];
    // one wave per workgroup: the lowest level is small
    const int tx = std::min(64, pow2ceil(g[3].n0)), ty = 64 / tx;
    const dim3 grid((g[3].n0 + tx - 1) / tx, (g[3].n1 + ty - 1) / ty, g[3].n2), block(tx, ty);
    using std::integral_constant;
    using X = integral_constant<int, 0>;
    using Y = integral_constant<int, 1>;
    using Z = integral_constant<int, 2>;
    switch (order) {
        case 1: launch(ch, grid, block, X(), Y(), Z()); break;
        case 2: launch(ch, grid, block, X(), Z(), Y()); break;
        case 3: launch(ch, grid, block, Y(), X(), Z()); break;
        case 5: launch(ch, grid, block, Y(), Z(), X()); break;
        case 6: launch(ch, grid, block, Z(), X(), Y()); break;
        default: launch(ch, grid, block, Z(), Y(), X()); break;
    }
}

template <typename T>
void launch_gather3(hipStream_t s, const Geo *g, int order, const T *const *pm, const T *const *pp, const T *r, T *fc) {
    launch_chain<T>(g, order, pm, pp, [&](const Chain<T> &ch, dim3 grid, dim3 block, auto a, auto b, auto c) {
        hipLaunchKernelGGL((k_gather3<T, a(), b(), c()>), grid, block, 0, s, ch, r, fc);
    });
}

template <typename T>
void launch_prolong3(hipStream_t s, const Geo *g, int order, const T *const *pm, const T *const *pp, const T *vc,
                     const T *vin, T *vout) {
    launch_chain<T>(g, order, pm, pp, [&](const Chain<T> &ch, dim3 grid, dim3 block, auto a, auto b, auto c) {
        hipLaunchKernelGGL((k_prolong3<T, a(), b(), c()>), grid, block, 0, s, ch, vc, vin, vout);
    });
}

template <typename Tin, typename Tout>
void launch_dense(hipStream_t s, int n, const double *Ainv, const Tin *f, Tout *v) {
    hipLaunchKernelGGL((k_dense_t<Tin, Tout>), dim3((n + 3) / 4), dim3(256), 0, s, n, Ainv, f, v);
}

template bool bottom_fits<double>(const Geo *, int);
template bool bottom_fits<float>(const Geo *, int);
template void launch_bottom<double>(hipStream_t, const BotArgs<double> &);
template void launch_bottom<float>(hipStream_t, const BotArgs<float> &);

#define INST(T)                                                                                                    \
    template void launch_apply<T>(hipStream_t, const Geo &, const T *, const T *, const T *, const T *, const T *, \
                                  T *, double *);                                                                  \
    template void launch_sweep<T>(hipStream_t, const Geo &, const T *, const T *, const T *, const T *, const T *, \
                                  const T *, T *, int, bool);                                                      \
    template void launch_sweep2<T>(hipStream_t, const Geo &, const T *, const T *, const T *, const T *,          \
                                   const T *, const T *, T *, int, bool);                                          \
    template void launch_smooth0<T>(hipStream_t, const Geo &, const T *, const T *, const T *, const T *,          \
                                    const T *, T *, int);                                                          \
    template void launch_resid<T>(hipStream_t, const Geo &, const T *, const T *, const T *, const T *, const T *, \
                                  const T *, T *);                                                                 \
    template void launch_gather<T>(hipStream_t, const Geo &, const Geo &, int, const T *, const T *, const T *,    \
                                   T *, bool);                                                                     \
    template void launch_prolong_to<T>(hipStream_t, const Geo &, const Geo &, int, const T *, const T *,           \
                                       const T *, const T *, T *, bool);                                           \
    template void launch_gather3<T>(hipStream_t, const Geo *, int, const T *const *, const T *const *, const T *,  \
                                    T *);                                                                          \
    template void launch_prolong3<T>(hipStream_t, const Geo *, int, const T *const *, const T *const *, const T *, \
                                     const T *, T *);                                                              \
    template void launch_dense<T, T>(hipStream_t, int, const double *, const T *, T *);
INST(double)
INST(float)
#undef INST

}  // namespace ngap
