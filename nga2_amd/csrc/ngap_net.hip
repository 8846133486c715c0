// Kernels of the small 3-D U-Net that supplies initial guesses and a
// flexible-PCG stage to the pressure solver (gfx950).
//
// Activations are channels-last: a[v][c], v = x + nx (y + ny z), BF16 for the
// convolution inputs, FP32 elsewhere. Padding is periodic (the workloads the
// network serves are periodic boxes). 3x3x3 convolutions are implicit GEMMs
// on BF16 MFMA (v_mfma_f32_16x16x32_bf16) with FP32 accumulation:
//   out[v][co] = sum_tap sum_ci W[tap][co][ci] * in[v + off(tap)][ci],
// tap = (dz+1)*9 + (dy+1)*3 + (dx+1), off = (dx, dy, dz) in {-1,0,1}^3.
// Weight layout [27][Cout][Cin] (ci fastest) makes both MFMA operands 16-byte
// LDS reads. Channel counts of MFMA layers are multiples of 32; the first
// layer (1-2 input channels) and the 1x1 output layer use plain FP32 kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ngapnet.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ int wrapi(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// Linear workgroup id remapped so that each of the 8 XCDs (workgroup b runs on
// XCD b % 8) walks one contiguous range: neighbouring tiles share the halo
// voxels in one L2. Bijective on [0, nb).
__device__ __forceinline__ int xcd_order(int b, int nb) {
    const int q = nb >> 3, r = nb & 7;
    const int x = b & 7, m = b >> 3;
    return x < r ? x * (q + 1) + m : r * (q + 1) + (x - r) * q + m;
}

// output tile of one workgroup: 16 x TY x 4 voxels, 4 waves (one z-slice each)
constexpr int TXV = 16, TYV = 4, TZV = 4;
constexpr int CK = 32;  // channel chunk

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- forward 3x3x3
// Implicit GEMM: M = 16 output channels (two blocks per workgroup), N = 16
// voxels along x, K = 32 input channels of one tap. A workgroup stages the halo
// tile of a 32-channel chunk in LDS, 64 bytes per voxel with the four 16-byte
// pieces rotated by (x / 2) % 4, so that the 16-byte reads of consecutive
// voxels fall on different banks without padding.
//
// With one LDS read per tap and operand the kernel was bound by the LDS read
// rate and by the staging between barriers. So a halo row is read once per
// (dz, dx) and used for the three taps dy of three output rows (TY + 2 reads
// for 6 TY MFMAs); the weights do not pass through LDS: each wave holds the nine
// taps of a plane dz and loads the next plane's from L1/L2, each into the
// registers of a tap that has done its last output row; and a workgroup walks
// over several tiles, with the next tile's (or chunk's) halo on its way to
// registers behind the products. TY = 8 takes 69 KB of LDS and 253 registers:
// two workgroups per CU. The sched_barriers keep the loads where they are
// written; the scheduler sinks them to their first use otherwise. D is
// transposed (weights as the first operand): a lane then holds four consecutive
// channels of a voxel and stores 8 (BF16) or 16 (FP32) bytes.
// An output sums its taps by chunk, dz, dy, dx. (With dy innermost, six taps of
// weights would do, and the figures below are 2 to 5% less; but another order
// flips the BF16 rounding of an output now and then, which a network's later
// layers turn into 3e-3 of its result.)
// 64 -> 32 channels at 128^3: 357 us (650 TFLOP/s) with 16 x 4 x 4 tiles and
// the weights staged in LDS, 266 us (870 TFLOP/s) now; 32 -> 64: 428 to 240 us
// (970 TFLOP/s). BF16 out, back to back.
// OFF: the type of a lane's byte offset within a plane of the input (32 bits
// unless a plane is 4 GB or more), added to an address held in scalar registers.
template <int TY, typename OFF>
__global__ void __launch_bounds__(256, 2) k_conv3_fwd(const __bf16 *__restrict__ in, const __bf16 *__restrict__ wt,
                                                      float *__restrict__ out32, __bf16 *__restrict__ outb, int nx,
                                                      int ny, int nz, int cin, int cout, int relu, int vst) {
    constexpr int HX = TXV + 2, HY = TY + 2, HZ = TZV + 2;
    constexpr int ROW = HX * CK, PL = HY * ROW;  // elements of one halo row and plane
    constexpr int NL = (HX * HY * 4 + 255) / 256;  // 16-byte pieces of a halo plane per thread
    __shared__ __attribute__((aligned(16))) __bf16 s_in[HZ * PL];
    const int tilesx = nx / TXV, tilesy = ny / TY, nco = cout / CK;
    const int ntiles = tilesx * tilesy * (nz / TZV) * nco;
    // tiles (channel block fastest) in one contiguous range per XCD (workgroup
    // b runs on XCD b % 8), so that neighbours share their halo in one L2
    const int nb = gridDim.x, xcd = blockIdx.x & 7, wgs = (nb + 7 - xcd) >> 3;
    const int before = xcd * (nb >> 3) + min(xcd, nb & 7);  // workgroups of the lower XCDs
    const int tfirst = (int)((long long)ntiles * before / nb) + (blockIdx.x >> 3);
    const int tend = (int)((long long)ntiles * (before + wgs) / nb);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const long long plane = (long long)nx * ny;
    // this lane's 16 bytes of a halo row for each x shift of the taps
    int xo[3];
#pragma unroll
    for (int dx = 0; dx < 3; dx++) xo[dx] = (lr + dx) * CK + ((lg ^ (((lr + dx) >> 1) & 3)) << 3);
    // LDS place of this thread's pieces (pieces past the plane repeat its last
    // voxel: the same bytes to the same place)
    int lx[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int hv = min((tid >> 2) + 64 * i, HX * HY - 1), hx = hv % HX;
        lx[i] = hv * CK + (((tid & 3) ^ ((hx >> 1) & 3)) << 3);
    }
    u32x4 rx[HZ][NL];
    // in-plane byte offsets of the pieces of tile t, then one halo plane of them
    OFF fo[NL];
    auto aim = [&](int t) {
        const int tt = t / nco;
        const int x0 = (tt % tilesx) * TXV, y0 = ((tt / tilesx) % tilesy) * TY;
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int hv = min((tid >> 2) + 64 * i, HX * HY - 1), hx = hv % HX, hy = hv / HX;
            fo[i] = (OFF)(wrapi(x0 - 1 + hx, nx) + nx * wrapi(y0 - 1 + hy, ny)) * (OFF)(2 * cin) + (tid & 3) * 16;
        }
        return (tt / (tilesx * tilesy)) * TZV;
    };
    auto fetch = [&](int z0, int ci0, int hz) {
        const char *b = reinterpret_cast<const char *>(in + wrapi(z0 - 1 + hz, nz) * plane * cin + ci0);
#pragma unroll
        for (int i = 0; i < NL; i++) rx[hz][i] = *reinterpret_cast<const u32x4 *>(b + fo[i]);
    };
    const long long wtap = (long long)cout * cin;
    const unsigned wo = (unsigned)(lr * cin + lg * 8) * 2u;
    bf16x8 w[3][3][2];
    // weights of tap (dz, dy, dx), two blocks of 16 channels, from the chunk's
    // (uniform) address wu
    auto wload = [&](const __bf16 *wu, int dz, int dy, int dx) {
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
            w[dy][dx][mb] = *reinterpret_cast<const bf16x8 *>(
                reinterpret_cast<const char *>(wu + (dz * 9 + dy * 3 + dx) * wtap + (long long)mb * 16 * cin) + wo);
    };
    auto chunk = [&](int t, int ci0) { return wt + (long long)(t % nco) * CK * cin + ci0; };
    f32x4 acc[TY][2];
    // one pass of the loop per 32-channel chunk of a tile: (t, ci0), then (tn, cn)
    int tn = tfirst, cn = 0;
    if (tn < tend) {
        const int z0 = aim(tn);
#pragma unroll
        for (int hz = 0; hz < HZ; hz++) fetch(z0, cn, hz);
#pragma unroll
        for (int dx = 0; dx < 3; dx++) wload(chunk(tn, cn), 0, 0, dx);
    }
    while (tn < tend) {
        const int t = tn, ci0 = cn;
        cn += CK;
        if (cn >= cin) {
            cn = 0;
            tn += wgs;
        }
        const int tt = t / nco;
        const int co0 = (t - tt * nco) * CK;
        if (ci0 == 0) {
#pragma unroll
            for (int a = 0; a < TY; a++)
#pragma unroll
                for (int b = 0; b < 2; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const int tc = min(tn, tend - 1);  // (behind the last chunk in vain)
        const __bf16 *wu = chunk(t, ci0), *wn = chunk(tc, cn);
        // (dy = 0 came with the previous chunk; more taps there, or none, measured slower)
#pragma unroll
        for (int q = 3; q < 9; q++) wload(wu, 0, q / 3, q % 3);
        __syncthreads();  // the previous chunk has been read
#pragma unroll
        for (int hz = 0; hz < HZ; hz++)
#pragma unroll
            for (int i = 0; i < NL; i++) *reinterpret_cast<u32x4 *>(s_in + hz * PL + lx[i]) = rx[hz][i];
        __syncthreads();
        const int zn = aim(tc);
        const __bf16 *base = s_in + PL * wave;
#pragma unroll
        for (int dz = 0; dz < 3; dz++) {
            bf16x8 a[3];
            a[0] = *reinterpret_cast<const bf16x8 *>(base + dz * PL + xo[0]);
            a[1] = *reinterpret_cast<const bf16x8 *>(base + dz * PL + xo[1]);
#pragma unroll
            for (int r = 0; r < HY; r++) {
                if (r == 2) fetch(zn, cn, 2 * dz);
                if (r == 4) fetch(zn, cn, 2 * dz + 1);
#pragma unroll
                for (int dx = 0; dx < 3; dx++) {
                    const int n = (dx + 2) % 3, rn = r + (dx + 2) / 3;  // two operands ahead
                    if (rn < HY) a[n] = *reinterpret_cast<const bf16x8 *>(base + dz * PL + rn * ROW + xo[n]);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int dy = 0; dy < 3; dy++) {
                        const int o = r - dy;
                        if (o < 0 || o >= TY) continue;
#pragma unroll
                        for (int mb = 0; mb < 2; mb++)
                            acc[o][mb] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[dy][dx][mb], a[dx], acc[o][mb], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // a tap that has done its last output row: the next plane's in its place
                    // (behind the last plane, the next chunk's first three)
                    if (dz < 2 ? r >= TY - 1 : r == TY - 1) {
                        wload(dz < 2 ? wu : wn, (dz + 1) % 3, r - (TY - 1), dx);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
        if (ci0 + CK < cin) continue;
        const int x0 = (tt % tilesx) * TXV, y0 = ((tt / tilesx) % tilesy) * TY, z0 = (tt / (tilesx * tilesy)) * TZV;
        // lane holds channels 4 lg + q of voxel lr of each 16 x 16 block
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        const unsigned lo = lr * cout + 4 * lg;
#pragma unroll
        for (int o = 0; o < TY; o++) {
            // the row's first element of this block (uniform)
            const long long e0 = (x0 + (long long)nx * ((y0 + o) + (long long)ny * (z0 + wave))) * cout + co0;
#pragma unroll
            for (int mb = 0; mb < 2; mb++) {
                const f32x4 d = acc[o][mb];
                if (out32) {
                    float *p = out32 + (e0 + mb * 16) + lo;
                    if (vst) {
                        *reinterpret_cast<f32x4 *>(p) = d;
                    } else {
                        for (int q = 0; q < 4; q++) p[q] = d[q];
                    }
                }
                if (outb) {
                    __bf16 *p = outb + (e0 + mb * 16) + lo;
                    bf16x4 b;
#pragma unroll
                    for (int q = 0; q < 4; q++) b[q] = (__bf16)(relu ? fmaxf(d[q], 0.f) : d[q]);
                    if (vst) {
                        *reinterpret_cast<bf16x4 *>(p) = b;
                    } else {
                        for (int q = 0; q < 4; q++) p[q] = b[q];
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// ---------------------------------------------------------------- weight gradient
// dW[tap][co][ci] = sum_v dout[v][co] * in[v + off(tap)][ci] as MFMA with K =
// voxels along x. Both operands lie in LDS as they lie in memory (channels
// fastest, 64 bytes per voxel) and are transposed by the read itself
// (ds_read_b64_tr_b16: a group of 16 lanes reads 4 voxels x 16 channels and
// lane i gets the 4 voxels of channel i), so an x shift is a voxel offset and
// nothing is scattered on the way in. The 32-byte halves of a voxel are
// exchanged by bit 1 of x, which spreads the reads over the banks.
//
// A wave owns one 16 x 16 block of (co, ci) for all 27 taps (108 accumulator
// registers); the 4 waves of a workgroup cover 32 x 32. A unit is a column of
// WX x 4 voxels over a range of planes: the workgroup marches over the input
// planes with the three dout planes that pair with each in a 4-deep ring and
// the next planes' loads in flight, one barrier per plane. Every input row is
// read once per dx and used for all (dy, dz): 30 operand reads for 108 MFMAs.
// part[p][cib][cob][27][32][32] holds the sums of workgroup p = 0 .. P-1.
// 64 -> 32 channels at 128^3: 848 us (scatter-transposed tiles, 274 TFLOP/s)
// before, 192 us (1210 TFLOP/s) now, and 97 against 11 us for the sum of the
// partials. WX = 32 needs nx % 32 == 0; WX = 16 uses the K = 16 MFMA, half its
// rate, and serves the rest.
constexpr int WY = 4;

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ s16x4 lds_tr(const __bf16 *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p);
}

template <int WX>
struct TrFrag;
template <>
struct TrFrag<32> {  // voxels 8 lg .. 8 lg + 7 of the row
    typedef bf16x8 type;
    static __device__ __forceinline__ type load(const __bf16 *p) {
        const s16x4 a = lds_tr(p), b = lds_tr(p + 4 * CK);
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        const s16x8 v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        return __builtin_bit_cast(bf16x8, v);
    }
    static __device__ __forceinline__ f32x4 mul(type a, type b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct TrFrag<16> {  // voxels 4 lg .. 4 lg + 3 of the row
    typedef s16x4 type;
    static __device__ __forceinline__ type load(const __bf16 *p) { return lds_tr(p); }
    static __device__ __forceinline__ f32x4 mul(type a, type b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
    }
};

template <int WX>
__global__ void __launch_bounds__(256, 2) k_conv3_wgrad(const __bf16 *__restrict__ in, const __bf16 *__restrict__ dout,
                                                        float *__restrict__ part, int nx, int ny, int nz, int cin,
                                                        int cout, int P, int zseg, int units) {
    typedef TrFrag<WX> F;
    constexpr int HXW = WX + 2, HYW = WY + 2;
    constexpr int XP = HYW * HXW * CK, DP = WY * WX * CK;  // elements of an input and a dout plane
    constexpr int NXL = (HYW * HXW * 4 + 255) / 256, NDL = WY * WX * 4 / 256;
    __shared__ __attribute__((aligned(16))) __bf16 s_x[2 * XP];
    __shared__ __attribute__((aligned(16))) __bf16 s_d[4 * DP];
    const int nob = cout / CK, nib = cin / CK;
    const int id = xcd_order(blockIdx.x, gridDim.x);
    const int blk = id / P, p = id - blk * P;
    const int cob = blk % nob, cib = blk / nob;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const int cb = wave & 1, ib = wave >> 1;
    f32x4 acc[27];
#pragma unroll
    for (int a = 0; a < 27; a++) acc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    // this lane's 8 bytes of a row: voxel x, half h of its channels
    auto voff = [](int x, int h) { return x * CK + ((h ^ ((x >> 1) & 1)) << 4); };
    const int xl = (WX / 4) * lg + (lr >> 2);
    const int ao = voff(xl, cb) + (lr & 3) * 4;
    int bo[3];
#pragma unroll
    for (int dx = 0; dx < 3; dx++) bo[dx] = voff(xl + dx, ib) + (lr & 3) * 4;
    const int colx = nx / WX, coly = ny / WY;
    const long long plane = (long long)nx * ny;
    for (int u = p; u < units; u += P) {
        const int c = u % (colx * coly);
        const int x0 = (c % colx) * WX, y0 = (c / colx) * WY;
        const int z0 = (u / (colx * coly)) * zseg, z1 = min(nz, z0 + zseg);
        // in-plane source and LDS place of this thread's pieces
        int gx[NXL], gd[NDL], lx[NXL], ld[NDL];
#pragma unroll
        for (int i = 0; i < NXL; i++) {
            // pieces past the plane repeat its last voxel (the same bytes to the same place)
            const int hv = min((tid >> 2) + 64 * i, HYW * HXW - 1), pc = tid & 3, hx = hv % HXW, hy = hv / HXW;
            gx[i] = wrapi(x0 - 1 + hx, nx) + nx * wrapi(y0 - 1 + hy, ny);
            lx[i] = hy * HXW * CK + voff(hx, pc >> 1) + (pc & 1) * 8;
        }
#pragma unroll
        for (int i = 0; i < NDL; i++) {
            const int hv = (tid >> 2) + 64 * i, pc = tid & 3, hx = hv % WX, hy = hv / WX;
            gd[i] = (x0 + hx) + nx * (y0 + hy);
            ld[i] = hy * WX * CK + voff(hx, pc >> 1) + (pc & 1) * 8;
        }
        u32x4 rx[NXL], rd[NDL];
        auto getx = [&](int hz) {
            const __bf16 *b = in + (long long)wrapi(hz, nz) * plane * cin + cib * CK + (tid & 3) * 8;
#pragma unroll
            for (int i = 0; i < NXL; i++) rx[i] = *reinterpret_cast<const u32x4 *>(b + (long long)gx[i] * cin);
        };
        // a dout plane that is not the unit's counts as zero
        auto getd = [&](int z) {
            const __bf16 *b = dout + (long long)min(z, z1 - 1) * plane * cout + cob * CK + (tid & 3) * 8;
#pragma unroll
            for (int i = 0; i < NDL; i++) rd[i] = *reinterpret_cast<const u32x4 *>(b + (long long)gd[i] * cout);
        };
        auto putx = [&](int hz) {
#pragma unroll
            for (int i = 0; i < NXL; i++) *reinterpret_cast<u32x4 *>(s_x + (hz & 1) * XP + lx[i]) = rx[i];
        };
        auto putd = [&](int z) {
#pragma unroll
            for (int i = 0; i < NDL; i++)
                *reinterpret_cast<u32x4 *>(s_d + (z & 3) * DP + ld[i]) = z < z1 ? rd[i] : u32x4{0u, 0u, 0u, 0u};
        };
        getx(z0 - 1);
        getd(z0);
        __syncthreads();  // the previous unit's planes have been read
        putx(z0 - 1);
        putd(z0);
        for (int q = 1; q < 3; q++)
#pragma unroll
            for (int i = 0; i < NDL; i++)
                *reinterpret_cast<u32x4 *>(s_d + ((z0 - q) & 3) * DP + ld[i]) = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
        for (int hz = z0 - 1; hz <= z1; hz++) {
            // the next planes, loaded behind this one's products (past the
            // unit's end loaded in vain)
            getx(min(hz + 1, z1));
            getd(hz + 2);
            const __bf16 *xp = s_x + (hz & 1) * XP;
            const __bf16 *dp[3];
#pragma unroll
            for (int dz = 0; dz < 3; dz++) dp[dz] = s_d + ((hz + 1 - dz) & 3) * DP + ao;
            // operands of a halo row one row ahead of its products; the
            // barriers keep the scheduler from hoisting all rows' reads, which
            // spills
            typename F::type A[3][WY], B[2][3];
            auto ldrow = [&](int hy) {
#pragma unroll
                for (int dx = 0; dx < 3; dx++) B[hy & 1][dx] = F::load(xp + hy * HXW * CK + bo[dx]);
                if (hy < WY) {
#pragma unroll
                    for (int dz = 0; dz < 3; dz++) A[dz][hy] = F::load(dp[dz] + hy * WX * CK);
                }
            };
            ldrow(0);
#pragma unroll
            for (int hy = 0; hy < HYW; hy++) {
                if (hy + 1 < HYW) ldrow(hy + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int dz = 0; dz < 3; dz++)
#pragma unroll
                    for (int dy = 0; dy < 3; dy++) {
                        const int y = hy - dy;
                        if (y < 0 || y >= WY) continue;
#pragma unroll
                        for (int dx = 0; dx < 3; dx++)
                            acc[dz * 9 + dy * 3 + dx] = F::mul(A[dz][y], B[hy & 1][dx], acc[dz * 9 + dy * 3 + dx]);
                    }
                __builtin_amdgcn_sched_barrier(0);
            }
            putx(hz + 1);
            putd(hz + 2);
            __syncthreads();
        }
    }
    // D[m = co][n = ci]: lane holds m = 4 lg + q, n = lr
    float *dst = part + (long long)((p * nib + cib) * nob + cob) * 27 * CK * CK;
#pragma unroll
    for (int t = 0; t < 27; t++)
#pragma unroll
        for (int q = 0; q < 4; q++) dst[(t * CK + cb * 16 + 4 * lg + q) * CK + ib * 16 + lr] = acc[t][q];
}

// dW[tap][co][ci] = sum_p part[p][cib][cob][tap][co%32][ci%32] in fixed order:
// a workgroup takes 64 consecutive entries of a partial, four slices of p per
// entry (p = s, s + 4, ...), and adds the slices in order. (One thread per
// entry over all partials was bound by the latency of its loads.)
__global__ void __launch_bounds__(256) k_wgrad_reduce(const float *__restrict__ part, float *__restrict__ dw, int cin,
                                                      int cout, int P) {
    __shared__ float sm[4][64];
    const int c = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const int n = 27 * cin * cout;  // entries of a partial; a multiple of 64
    const int e = blockIdx.x * 64 + c;
    float s = 0.f;
#pragma unroll 8
    for (int p = sl; p < P; p += 4) s += part[(long long)p * n + e];
    sm[sl][c] = s;
    __syncthreads();
    if (sl == 0) {
        const int ci = e % CK, co = (e / CK) % CK, tap = (e / (CK * CK)) % 27, blk = e / (27 * CK * CK);
        const int nob = cout / CK, cob = blk % nob, cib = blk / nob;
        dw[((long long)tap * cout + cob * CK + co) * cin + cib * CK + ci] =
            (sm[0][c] + sm[1][c]) + (sm[2][c] + sm[3][c]);
    }
}

// weights of the data gradient: wd[tap'][ci][co] = wt[26 - tap'][co][ci]
__global__ void k_flip_transpose(const __bf16 *__restrict__ wt, __bf16 *__restrict__ wd, int cin, int cout) {
    const long long n = 27LL * cin * cout;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int co = (int)(i % cout);
        const int ci = (int)((i / cout) % cin);
        const int tp = (int)(i / ((long long)cin * cout));
        wd[i] = wt[((long long)(26 - tp) * cout + co) * cin + ci];
    }
}

// ---------------------------------------------------------------- small-channel layers (FP32)
// out[v][co] = sum_tap sum_ci w[tap][co][ci] in[v+off][ci]   (cin small)
__global__ void k_conv3_small_fwd(const float *__restrict__ in, const float *__restrict__ w, float *__restrict__ out32,
                                  __bf16 *__restrict__ outb, int nx, int ny, int nz, int cin, int cout, int relu) {
    const long long nv = (long long)nx * ny * nz;
    const long long i = blockIdx.x * 256LL + threadIdx.x;
    if (i >= nv * cout) return;
    const int co = (int)(i % cout);
    const long long v = i / cout;
    const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long long)nx * ny));
    float s = 0.f;
    for (int tap = 0; tap < 27; tap++) {
        const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
        const long long u = wrapi(x + dx, nx) + (long long)nx * (wrapi(y + dy, ny) + (long long)ny * wrapi(z + dz, nz));
        for (int ci = 0; ci < cin; ci++) s += w[(tap * cout + co) * cin + ci] * in[u * cin + ci];
    }
    if (out32) out32[i] = s;
    if (outb) outb[i] = (__bf16)(relu ? fmaxf(s, 0.f) : s);
}

// The first layer (one input channel): one thread per voxel computes all COUT
// outputs from its 27 input values, with the weights in LDS (a broadcast read
// per tap and channel), and writes the voxel's COUT channels as 16-byte
// stores. Same summation order per output as k_conv3_small_fwd (taps in
// order). The per-(voxel, channel) form re-read the 27 inputs for every
// channel and spent its time in index arithmetic.
template <int COUT>
__global__ void __launch_bounds__(256) k_conv3_c1_fwd(const float *__restrict__ in, const float *__restrict__ w,
                                                      float *__restrict__ out32, __bf16 *__restrict__ outb, int nx,
                                                      int ny, int nz, int relu) {
    __shared__ float sw[27 * COUT];
    for (int q = threadIdx.x; q < 27 * COUT; q += 256) sw[q] = w[q];
    __syncthreads();
    const int nv = nx * ny * nz;
    const int v = blockIdx.x * 256 + threadIdx.x;
    if (v >= nv) return;
    const int x = v % nx, y = (v / nx) % ny, z = v / (nx * ny);
    float acc[COUT];
#pragma unroll
    for (int co = 0; co < COUT; co++) acc[co] = 0.f;
#pragma unroll
    for (int tap = 0; tap < 27; tap++) {
        const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
        const float iv = in[wrapi(x + dx, nx) + nx * (wrapi(y + dy, ny) + ny * wrapi(z + dz, nz))];
#pragma unroll
        for (int co = 0; co < COUT; co++) acc[co] += sw[tap * COUT + co] * iv;
    }
    const long long o = (long long)v * COUT;
    if (out32) {
#pragma unroll
        for (int co = 0; co < COUT; co += 4)
            *reinterpret_cast<float4 *>(out32 + o + co) = make_float4(acc[co], acc[co + 1], acc[co + 2], acc[co + 3]);
    }
    if (outb) {
#pragma unroll
        for (int co = 0; co < COUT; co += 8) {
            bf16x8 b;
#pragma unroll
            for (int q = 0; q < 8; q++) b[q] = (__bf16)(relu ? fmaxf(acc[co + q], 0.f) : acc[co + q]);
            *reinterpret_cast<bf16x8 *>(outb + o + co) = b;
        }
    }
}

// dW of the small layer: one block per weight, fixed-order block reduction
__global__ void __launch_bounds__(256) k_conv3_small_wgrad(const float *__restrict__ in, const float *__restrict__ dout,
                                                           float *__restrict__ dw, int nx, int ny, int nz, int cin,
                                                           int cout) {
    __shared__ float sm[4];
    const int wi = blockIdx.x;  // tap*cout*cin + co*cin + ci
    const int ci = wi % cin, co = (wi / cin) % cout, tap = wi / (cin * cout);
    const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
    const long long nv = (long long)nx * ny * nz;
    float s = 0.f;
    for (long long v = threadIdx.x; v < nv; v += 256) {
        const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long long)nx * ny));
        const long long u = wrapi(x + dx, nx) + (long long)nx * (wrapi(y + dy, ny) + (long long)ny * wrapi(z + dz, nz));
        s += dout[v * cout + co] * in[u * cin + ci];
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) dw[wi] = sm[0] + sm[1] + sm[2] + sm[3];
}

// dW of a 1-input-channel layer over bricks of 32 x 8 x 8 voxels: the brick's
// input with a one-voxel halo sits in LDS, thread (voxel column vx, channel
// quad q) accumulates all 27 taps of its 4 channels (108 registers), so dout
// is read once, as one 16-byte load per thread and voxel. Partial bricks at
// the upper faces skip the voxels beyond the grid. Partials per workgroup,
// part[b][tap][co], summed in fixed order by k_colsum.
constexpr int SW_BLOCKS = 1024;
constexpr int SB_X = 32, SB_Y = 8, SB_Z = 8;
constexpr int SB_HX = SB_X + 2, SB_HY = SB_Y + 2, SB_HZ = SB_Z + 2;

template <int COUT>
__global__ void __launch_bounds__(256) k_small_wgrad_brick(const float *__restrict__ in, const float *__restrict__ dout,
                                                           float *__restrict__ part, int nx, int ny, int nz) {
    constexpr int NQ = COUT / 4;
    static_assert(256 / NQ == SB_X, "one voxel column per thread group");
    __shared__ float s_in[SB_HX * SB_HY * SB_HZ];
    __shared__ float s_red[4][27 * COUT];
    const int tid = threadIdx.x, q = tid % NQ, vx = tid / NQ;
    const int nbx = (nx + SB_X - 1) / SB_X, nby = (ny + SB_Y - 1) / SB_Y, nbz = (nz + SB_Z - 1) / SB_Z;
    const int nb = nbx * nby * nbz;
    float acc[27][4];
#pragma unroll
    for (int t = 0; t < 27; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[t][k] = 0.f;
    for (int brick = blockIdx.x; brick < nb; brick += gridDim.x) {
        const int x0 = (brick % nbx) * SB_X, y0 = ((brick / nbx) % nby) * SB_Y, z0 = (brick / (nbx * nby)) * SB_Z;
        __syncthreads();
        // halo coordinates beyond n are clamped to n: only voxels inside the
        // grid are accumulated, and they read at most one past the last
        for (int i = tid; i < SB_HX * SB_HY * SB_HZ; i += 256) {
            const int hx = i % SB_HX, hy = (i / SB_HX) % SB_HY, hz = i / (SB_HX * SB_HY);
            const int gx = wrapi(min(x0 - 1 + hx, nx), nx), gy = wrapi(min(y0 - 1 + hy, ny), ny),
                      gz = wrapi(min(z0 - 1 + hz, nz), nz);
            s_in[i] = in[gx + (long long)nx * (gy + (long long)ny * gz)];
        }
        __syncthreads();
        if (x0 + vx >= nx) continue;
        const int ly1 = min(SB_Y, ny - y0), lz1 = min(SB_Z, nz - z0);
        for (int lz = 0; lz < lz1; lz++)
            for (int ly = 0; ly < ly1; ly++) {
                const long long v = (x0 + vx) + (long long)nx * ((y0 + ly) + (long long)ny * (z0 + lz));
                const float4 d = reinterpret_cast<const float4 *>(dout + v * COUT)[q];
#pragma unroll
                for (int t = 0; t < 27; t++) {
                    const float x = s_in[(vx + t % 3) + SB_HX * ((ly + (t / 3) % 3) + SB_HY * (lz + t / 9))];
                    acc[t][0] += d.x * x;
                    acc[t][1] += d.y * x;
                    acc[t][2] += d.z * x;
                    acc[t][3] += d.w * x;
                }
            }
    }
    // lanes with the same channel quad: lane % NQ; sum over the wave, then the 4 waves
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int t = 0; t < 27; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float r = acc[t][k];
            for (int off = NQ; off < 64; off <<= 1) r += __shfl_xor(r, off, 64);
            if (lane < NQ) s_red[wave][t * COUT + 4 * q + k] = r;
        }
    __syncthreads();
    for (int i = tid; i < 27 * COUT; i += 256)
        part[(long long)blockIdx.x * 27 * COUT + i] = s_red[0][i] + s_red[1][i] + s_red[2][i] + s_red[3][i];
}

// out[i] = sum_b part[b][i], i < n: workgroup of 16 columns x 16 slices, slice
// s sums b = s, s + 16, ... and the 16 slice sums are added in slice order
__global__ void __launch_bounds__(256) k_colsum(const float *__restrict__ part, float *__restrict__ out, int nb, int n) {
    __shared__ float sm[16][17];
    const int c = threadIdx.x & 15, sl = threadIdx.x >> 4;
    const int i = blockIdx.x * 16 + c;
    float s = 0.f;
    if (i < n)
        for (int b = sl; b < nb; b += 16) s += part[(long long)b * n + i];
    sm[sl][c] = s;
    __syncthreads();
    if (sl == 0 && i < n) {
        float t = 0.f;
        for (int k = 0; k < 16; k++) t += sm[k][c];
        out[i] = t;
    }
}

// dx[v][c] = w[c] dy[v]; dW partials per block (C known at compile time, registers only)
template <int C>
__global__ void __launch_bounds__(256) k_conv1_bwd_t(const __bf16 *__restrict__ x, const float *__restrict__ w,
                                                     const float *__restrict__ dy, float *__restrict__ dx,
                                                     float *__restrict__ part, long long nv) {
    __shared__ float sm[4][C];
    float accw[C];
    float wr[C];
#pragma unroll
    for (int ch = 0; ch < C; ch++) {
        accw[ch] = 0.f;
        wr[ch] = w[ch];
    }
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < nv; v += (long long)gridDim.x * 256) {
        const float g = dy[v];
#pragma unroll
        for (int ch = 0; ch < C; ch++) {
            dx[v * C + ch] = wr[ch] * g;
            accw[ch] += g * (float)x[v * C + ch];
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int ch = 0; ch < C; ch++) {
        float t = accw[ch];
        for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
        if (lane == 0) sm[wave][ch] = t;
    }
    __syncthreads();
    if (threadIdx.x < C)
        part[blockIdx.x * C + threadIdx.x] = sm[0][threadIdx.x] + sm[1][threadIdx.x] + sm[2][threadIdx.x] + sm[3][threadIdx.x];
}

// ---------------------------------------------------------------- elementwise
__global__ void k_relu_bwd(const float *__restrict__ dy, const __bf16 *__restrict__ y, float *__restrict__ dx,
                           __bf16 *__restrict__ dxb, long long n) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float g = (float)y[i] > 0.f ? dy[i] : 0.f;
        if (dx) dx[i] = g;
        if (dxb) dxb[i] = (__bf16)g;
    }
}

// The same in pieces of 4 (n % 4 == 0, dy/dx 16-byte and y/dxb 8-byte aligned)
__global__ void k_relu_bwd_v4(const float *__restrict__ dy, const __bf16 *__restrict__ y, float *__restrict__ dx,
                              __bf16 *__restrict__ dxb, long long n4) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n4; i += (long long)gridDim.x * 256) {
        const float4 d = reinterpret_cast<const float4 *>(dy)[i];
        const bf16x4 yv = reinterpret_cast<const bf16x4 *>(y)[i];
        const float4 g = make_float4((float)yv[0] > 0.f ? d.x : 0.f, (float)yv[1] > 0.f ? d.y : 0.f,
                                     (float)yv[2] > 0.f ? d.z : 0.f, (float)yv[3] > 0.f ? d.w : 0.f);
        if (dx) reinterpret_cast<float4 *>(dx)[i] = g;
        if (dxb) {
            bf16x4 b;
            b[0] = (__bf16)g.x;
            b[1] = (__bf16)g.y;
            b[2] = (__bf16)g.z;
            b[3] = (__bf16)g.w;
            reinterpret_cast<bf16x4 *>(dxb)[i] = b;
        }
    }
}

__global__ void k_to_bf16(const float *__restrict__ s, __bf16 *__restrict__ d, long long n) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) d[i] = (__bf16)s[i];
}

// average pool 2x2x2 (bf16 -> bf16), fine dims nx,ny,nz
__global__ void k_pool2(const __bf16 *__restrict__ in, __bf16 *__restrict__ out, int nx, int ny, int nz, int c) {
    const int mx = nx / 2, my = ny / 2, mz = nz / 2;
    const long long n = (long long)mx * my * mz * c;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int ch = (int)(i % c);
        const long long v = i / c;
        const int x = (int)(v % mx), y = (int)((v / mx) % my), z = (int)(v / ((long long)mx * my));
        float s = 0.f;
        for (int q = 0; q < 8; q++) {
            const long long u = (2 * x + (q & 1)) + (long long)nx * ((2 * y + ((q >> 1) & 1)) + (long long)ny * (2 * z + (q >> 2)));
            s += (float)in[u * c + ch];
        }
        out[i] = (__bf16)(0.125f * s);
    }
}

// The same in pieces of 8 channels (c % 8 == 0, 16-byte aligned). With cat, the
// input also goes into the channels d0 .. d0 + c of a concatenation buffer of
// ctot channels (even nx, ny, nz: every voxel belongs to a pool window), which
// saves the pass that read it again. Bound by memory: the three pools and copies of
// a forward pass at 128^3 took 61 (scalar pool) and 59 us, 68 us now.
__global__ void __launch_bounds__(256) k_pool2_v8(const __bf16 *__restrict__ in, __bf16 *__restrict__ out,
                                                  __bf16 *__restrict__ cat, int nx, int ny, int nz, int c, int ctot,
                                                  int d0) {
    const int mx = nx / 2, my = ny / 2, mz = nz / 2, c8 = c / 8;
    const long long n = (long long)mx * my * mz * c8;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int g = (int)(i % c8);
        const long long v = i / c8, r = v / mx;
        const int x = (int)(v - r * mx), y = (int)(r % my), z = (int)(r / my);
        bf16x8 p[8];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const long long u = (2 * x + (q & 1)) + (long long)nx * ((2 * y + ((q >> 1) & 1)) + (long long)ny * (2 * z + (q >> 2)));
            p[q] = *reinterpret_cast<const bf16x8 *>(in + u * c + 8 * g);
        }
        float s[8] = {};
#pragma unroll
        for (int q = 0; q < 8; q++) {
#pragma unroll
            for (int e = 0; e < 8; e++) s[e] += (float)p[q][e];
            if (cat) {
                const long long u = (2 * x + (q & 1)) + (long long)nx * ((2 * y + ((q >> 1) & 1)) + (long long)ny * (2 * z + (q >> 2)));
                *reinterpret_cast<bf16x8 *>(cat + u * ctot + d0 + 8 * g) = p[q];
            }
        }
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = (__bf16)(0.125f * s[e]);
        *reinterpret_cast<bf16x8 *>(out + i * 8) = o;
    }
}

// d(in) of the pool: each fine voxel gets dout(coarse)/8 (fp32 -> fp32, added to dst when acc)
__global__ void k_pool2_bwd(const float *__restrict__ dout, float *__restrict__ din, int nx, int ny, int nz, int c,
                            int acc) {
    const long long n = (long long)nx * ny * nz * c;
    const int mx = nx / 2, my = ny / 2;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int ch = (int)(i % c);
        const long long v = i / c;
        const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long long)nx * ny));
        const long long u = (x / 2) + (long long)mx * ((y / 2) + (long long)my * (z / 2));
        const float g = 0.125f * dout[u * c + ch];
        din[i] = acc ? din[i] + g : g;
    }
}

// The same in pieces of 4 channels (c % 4 == 0)
__global__ void k_pool2_bwd_v4(const float *__restrict__ dout, float *__restrict__ din, int nx, int ny, int nz, int c,
                               int acc) {
    const int c4 = c / 4;
    const long long n = (long long)nx * ny * nz * c4;
    const int mx = nx / 2, my = ny / 2;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int g4 = (int)(i % c4);
        const long long v = i / c4;
        const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long long)nx * ny));
        const long long u = (x / 2) + (long long)mx * ((y / 2) + (long long)my * (z / 2));
        const float4 d = *reinterpret_cast<const float4 *>(dout + u * c + 4 * g4);
        float4 g = make_float4(0.125f * d.x, 0.125f * d.y, 0.125f * d.z, 0.125f * d.w);
        float4 *o = reinterpret_cast<float4 *>(din) + i;
        if (acc) {
            const float4 p = *o;
            g = make_float4(p.x + g.x, p.y + g.y, p.z + g.z, p.w + g.w);
        }
        *o = g;
    }
}

// out[fine][c0 + ch] = in[coarse][ch] (nearest-neighbour upsampling into a
// channel slice of a concatenation buffer with ctot channels)
__global__ void k_up2(const __bf16 *__restrict__ in, __bf16 *__restrict__ out, int nx, int ny, int nz, int c, int ctot,
                      int c0) {
    const long long n = (long long)nx * ny * nz * c;
    const int mx = nx / 2, my = ny / 2;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int ch = (int)(i % c);
        const long long v = i / c;
        const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long long)nx * ny));
        const long long u = (x / 2) + (long long)mx * ((y / 2) + (long long)my * (z / 2));
        out[v * ctot + c0 + ch] = in[u * c + ch];
    }
}

// The same copy in 16-byte pieces of 8 channels (c, ctot, c0 multiples of 8)
__global__ void k_up2_v8(const __bf16 *__restrict__ in, __bf16 *__restrict__ out, int nx, int ny, int nz, int c,
                         int ctot, int c0) {
    const int c8 = c / 8;
    const long long n = (long long)nx * ny * nz * c8;
    const int mx = nx / 2, my = ny / 2;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int g = (int)(i % c8);
        const long long v = i / c8;
        const int x = (int)(v % nx), y = (int)((v / nx) % ny), z = (int)(v / ((long long)nx * ny));
        const long long u = (x / 2) + (long long)mx * ((y / 2) + (long long)my * (z / 2));
        *reinterpret_cast<bf16x8 *>(out + v * ctot + c0 + 8 * g) = *reinterpret_cast<const bf16x8 *>(in + u * c + 8 * g);
    }
}

// d(coarse) = sum over the 8 fine children of d(fine)[c0 + ch]
__global__ void k_up2_bwd(const float *__restrict__ dout, float *__restrict__ din, int nx, int ny, int nz, int c,
                          int ctot, int c0) {
    const int mx = nx / 2, my = ny / 2, mz = nz / 2;
    const long long n = (long long)mx * my * mz * c;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int ch = (int)(i % c);
        const long long v = i / c;
        const int x = (int)(v % mx), y = (int)((v / mx) % my), z = (int)(v / ((long long)mx * my));
        float s = 0.f;
        for (int q = 0; q < 8; q++) {
            const long long u = (2 * x + (q & 1)) + (long long)nx * ((2 * y + ((q >> 1) & 1)) + (long long)ny * (2 * z + (q >> 2)));
            s += dout[u * ctot + c0 + ch];
        }
        din[i] = s;
    }
}

// The same in pieces of 4 channels (c, ctot, c0 multiples of 4)
__global__ void k_up2_bwd_v4(const float *__restrict__ dout, float *__restrict__ din, int nx, int ny, int nz, int c,
                             int ctot, int c0) {
    const int mx = nx / 2, my = ny / 2, mz = nz / 2, c4 = c / 4;
    const long long n = (long long)mx * my * mz * c4;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int g4 = (int)(i % c4);
        const long long v = i / c4;
        const int x = (int)(v % mx), y = (int)((v / mx) % my), z = (int)(v / ((long long)mx * my));
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int q = 0; q < 8; q++) {
            const long long u = (2 * x + (q & 1)) + (long long)nx * ((2 * y + ((q >> 1) & 1)) + (long long)ny * (2 * z + (q >> 2)));
            const float4 d = *reinterpret_cast<const float4 *>(dout + u * ctot + c0 + 4 * g4);
            s.x += d.x;
            s.y += d.y;
            s.z += d.z;
            s.w += d.w;
        }
        reinterpret_cast<float4 *>(din)[i] = s;
    }
}

// copy a channel slice: dst[v][d0 + ch] = src[v][s0 + ch], ch < c (bf16 or fp32)
// the same copy in 16-byte pieces (c, cs, s0, cd, d0 multiples of 16 / sizeof(T))
template <typename T>
__global__ void k_chan_copy_v16(const T *__restrict__ src, T *__restrict__ dst, long long nv, int c, int cs, int s0,
                                int cd, int d0) {
    constexpr int E = 16 / sizeof(T);
    const int ce = c / E;
    const long long n = nv * ce;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int g = (int)(i % ce);
        const long long v = i / ce;
        *reinterpret_cast<uint4 *>(dst + v * cd + d0 + g * E) = *reinterpret_cast<const uint4 *>(src + v * cs + s0 + g * E);
    }
}

template <typename T>
__global__ void k_chan_copy(const T *__restrict__ src, T *__restrict__ dst, long long nv, int c, int cs, int s0, int cd,
                            int d0) {
    const long long n = nv * c;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int ch = (int)(i % c);
        const long long v = i / c;
        dst[v * cd + d0 + ch] = src[v * cs + s0 + ch];
    }
}

// y[v] = sum_c w[c] x[v][c] (1x1 output layer, x bf16)
// y[v] = sum_ch w[ch] x[v][ch] for C channels: one thread per voxel reading its
// C bf16 values as 16-byte loads (C a multiple of 8), channels summed in order
template <int C>
__global__ void __launch_bounds__(256) k_conv1_fwd_t(const __bf16 *__restrict__ x, const float *__restrict__ w,
                                                     float *__restrict__ y, long long nv) {
    float wr[C];
#pragma unroll
    for (int ch = 0; ch < C; ch++) wr[ch] = w[ch];
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < nv; v += (long long)gridDim.x * 256) {
        float s = 0.f;
#pragma unroll
        for (int c8 = 0; c8 < C; c8 += 8) {
            const bf16x8 b = *reinterpret_cast<const bf16x8 *>(x + v * C + c8);
#pragma unroll
            for (int q = 0; q < 8; q++) s += wr[c8 + q] * (float)b[q];
        }
        y[v] = s;
    }
}

__global__ void k_conv1_fwd(const __bf16 *__restrict__ x, const float *__restrict__ w, float *__restrict__ y,
                            long long nv, int c) {
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < nv; v += (long long)gridDim.x * 256) {
        float s = 0.f;
        for (int ch = 0; ch < c; ch++) s += w[ch] * (float)x[v * c + ch];
        y[v] = s;
    }
}

// dx[v][c] = w[c] dy[v]; dW partials per block: part[b][c] = sum_v dy[v] x[v][c]
__global__ void __launch_bounds__(256) k_conv1_bwd(const __bf16 *__restrict__ x, const float *__restrict__ w,
                                                   const float *__restrict__ dy, float *__restrict__ dx,
                                                   float *__restrict__ part, long long nv, int c) {
    __shared__ float sm[4][64];
    float accw[64];
    for (int ch = 0; ch < c; ch++) accw[ch] = 0.f;
    for (long long v = blockIdx.x * 256LL + threadIdx.x; v < nv; v += (long long)gridDim.x * 256) {
        const float g = dy[v];
        for (int ch = 0; ch < c; ch++) {
            dx[v * c + ch] = w[ch] * g;
            accw[ch] += g * (float)x[v * c + ch];
        }
    }
    for (int ch = 0; ch < c; ch++) {
        float s = accw[ch];
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6][ch] = s;
    }
    __syncthreads();
    if (threadIdx.x < c) part[blockIdx.x * c + threadIdx.x] = sm[0][threadIdx.x] + sm[1][threadIdx.x] + sm[2][threadIdx.x] + sm[3][threadIdx.x];
}

// Adam on FP32 master weights; writes the BF16 copy
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m, float *__restrict__ v,
                       __bf16 *__restrict__ wb, long long n, float lr, float b1, float b2, float eps, float c1,
                       float c2, float scale) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float gi = g[i] * scale;
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        w[i] = wi;
        if (wb) wb[i] = (__bf16)wi;
    }
}

int blocks_for(long long n) {
    long long b = (n + 255) / 256;
    if (b > 16384) b = 16384;
    return (int)(b < 1 ? 1 : b);
}

template <typename T>
int chan_copy(const T *src, T *dst, long long nv, int c, int cs, int s0, int cd, int d0, void *stream) {
    constexpr int E = 16 / sizeof(T);
    if ((c | cs | s0 | cd | d0) % E == 0 && ((uintptr_t)src | (uintptr_t)dst) % 16 == 0)
        hipLaunchKernelGGL(k_chan_copy_v16<T>, dim3(blocks_for(nv * c / E)), dim3(256), 0, (hipStream_t)stream, src,
                           dst, nv, c, cs, s0, cd, d0);
    else
        hipLaunchKernelGGL(k_chan_copy<T>, dim3(blocks_for(nv * c)), dim3(256), 0, (hipStream_t)stream, src, dst, nv,
                           c, cs, s0, cd, d0);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// boxes and channel counts that the tiled convolutions take
bool tiled(int nx, int ny, int nz, int cin, int cout) {
    return nx > 0 && ny > 0 && nz > 0 && cin > 0 && cout > 0 && nx % TXV == 0 && ny % TYV == 0 && nz % TZV == 0 &&
           cin % CK == 0 && cout % CK == 0;
}

}  // namespace

extern "C" {

int ngapnet_conv3_fwd(const void *in, const void *wt, float *out32, void *outb, int nx, int ny, int nz, int cin,
                      int cout, int relu, void *stream) {
    if (!tiled(nx, ny, nz, cin, cout)) return -1;
    const int vst = (uintptr_t)out32 % 16 == 0 && (uintptr_t)outb % 8 == 0;
    const long long wg4 = (long long)(nx / TXV) * (ny / TYV) * (nz / TZV) * (cout / CK);
    // 16 x 8 x 4 tiles where they still give every CU a workgroup; smaller
    // grids take 16 x 4 x 4 so that the chip is not left idle. At most two
    // workgroups per CU are launched; they walk over the tiles.
    const auto wgs = [](long long tiles) { return dim3((unsigned)(tiles < 512 ? tiles : 512)); };
    const bool big = (long long)nx * ny * cin * 2 >= (1LL << 32);
    if (big)
        hipLaunchKernelGGL((k_conv3_fwd<4, unsigned long long>), wgs(wg4), dim3(256), 0, (hipStream_t)stream,
                           (const __bf16 *)in, (const __bf16 *)wt, out32, (__bf16 *)outb, nx, ny, nz, cin, cout, relu,
                           vst);
    else if (ny % 8 == 0 && wg4 / 2 >= 256)
        hipLaunchKernelGGL((k_conv3_fwd<8, unsigned>), wgs(wg4 / 2), dim3(256), 0, (hipStream_t)stream,
                           (const __bf16 *)in, (const __bf16 *)wt, out32, (__bf16 *)outb, nx, ny, nz, cin, cout, relu,
                           vst);
    else
        hipLaunchKernelGGL((k_conv3_fwd<4, unsigned>), wgs(wg4), dim3(256), 0, (hipStream_t)stream, (const __bf16 *)in,
                           (const __bf16 *)wt, out32, (__bf16 *)outb, nx, ny, nz, cin, cout, relu, vst);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_wgrad_parts(int nx, int ny, int nz, int cin, int cout) {
    const int ntiles = (nx / TXV) * (ny / TYV) * (nz / TZV);
    int G = ntiles < 256 ? ntiles : 256;
    (void)cin;
    (void)cout;
    return G;
}

int ngapnet_conv3_wgrad(const void *in, const void *dout, float *dw, float *part, int nx, int ny, int nz, int cin,
                        int cout, void *stream) {
    if (!tiled(nx, ny, nz, cin, cout)) return -1;
    const int blocks = (cin / CK) * (cout / CK);
    const int wx = nx % 32 == 0 ? 32 : 16;
    const int cols = (nx / wx) * (ny / WY);
    const int G = ngapnet_wgrad_parts(nx, ny, nz, cin, cout);
    // workgroups per 32 x 32 channel block: two per CU over all blocks; columns
    // are cut into ranges of planes (at least 4: each range reads two more) until
    // there is a unit for each
    const int W = std::max(1, std::min(G, 512 / blocks));
    int nseg = std::min((W + cols - 1) / cols, nz / 4);
    // ... and into shorter ranges where a partial would be a longer chain of FP32
    // sums than 256 partials need. The 2-norm error of dW is about
    // 2^-24 sqrt(L / 4 + G / 11) for G partials of L products of 32 voxels added
    // one after the other; here those are added in four slices, so that L may be
    // G / 4 more. Against 64 bits, with 256 partials, with one per workgroup (the
    // fewer the more channel blocks), and now: 64^3, 128 -> 128 channels 3.2e-7,
    // 4.8e-7 (185 us), 2.7e-7 (250 us); 128^3, 96 -> 32 5.7e-7, 6.8e-7 (340 us),
    // 5.1e-7 (300 us).
    const long long tiles = (long long)(nx / TXV) * (ny / TYV) * (nz / TZV);
    const long long most = 256 * ((tiles + G - 1) / G) + 8LL * G;  // voxels of a partial
    const int zmax = (int)std::max(1LL, std::min((long long)nz, most / (WY * wx)));
    nseg = std::max(nseg, (nz + zmax - 1) / zmax);
    const int zseg = (nz + nseg - 1) / nseg;
    nseg = (nz + zseg - 1) / zseg;
    const int units = cols * nseg;
    // units of a partial; more partials than W run as further workgroups
    const int each = (int)std::max(1LL, most / ((long long)zseg * WY * wx));
    const int P = std::min(std::min(G, units), std::max(W, (units + each - 1) / each));
    const dim3 grid((unsigned)(P * blocks));
    if (wx == 32)
        hipLaunchKernelGGL(k_conv3_wgrad<32>, grid, dim3(256), 0, (hipStream_t)stream, (const __bf16 *)in,
                           (const __bf16 *)dout, part, nx, ny, nz, cin, cout, P, zseg, units);
    else
        hipLaunchKernelGGL(k_conv3_wgrad<16>, grid, dim3(256), 0, (hipStream_t)stream, (const __bf16 *)in,
                           (const __bf16 *)dout, part, nx, ny, nz, cin, cout, P, zseg, units);
    hipLaunchKernelGGL(k_wgrad_reduce, dim3((unsigned)(27 * cin * cout / 64)), dim3(256), 0, (hipStream_t)stream,
                       (const float *)part, dw, cin, cout, P);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_flip_transpose(const void *wt, void *wd, int cin, int cout, void *stream) {
    hipLaunchKernelGGL(k_flip_transpose, dim3(blocks_for(27LL * cin * cout)), dim3(256), 0, (hipStream_t)stream,
                       (const __bf16 *)wt, (__bf16 *)wd, cin, cout);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_conv3_small_fwd(const float *in, const float *w, float *out32, void *outb, int nx, int ny, int nz,
                            int cin, int cout, int relu, void *stream) {
    const long long nv = (long long)nx * ny * nz;
    if (cin == 1 && cout == 32 && nv < (1LL << 31)) {
        hipLaunchKernelGGL(k_conv3_c1_fwd<32>, dim3((unsigned)((nv + 255) / 256)), dim3(256), 0, (hipStream_t)stream, in,
                           w, out32, (__bf16 *)outb, nx, ny, nz, relu);
        return hipGetLastError() == hipSuccess ? 0 : 1;
    }
    const long long n = nv * cout;
    hipLaunchKernelGGL(k_conv3_small_fwd, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, in, w,
                       out32, (__bf16 *)outb, nx, ny, nz, cin, cout, relu);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_conv3_small_wgrad(const float *in, const float *dout, float *dw, float *part, int nx, int ny, int nz,
                              int cin, int cout, void *stream) {
    if (part && cin == 1 && cout == 32 && (uintptr_t)dout % 16 == 0) {
        const long long bricks = (long long)((nx + SB_X - 1) / SB_X) * ((ny + SB_Y - 1) / SB_Y) * ((nz + SB_Z - 1) / SB_Z);
        const int grid = (int)(bricks < SW_BLOCKS ? bricks : SW_BLOCKS);
        hipLaunchKernelGGL(k_small_wgrad_brick<32>, dim3(grid), dim3(256), 0, (hipStream_t)stream, in, dout, part, nx,
                           ny, nz);
        hipLaunchKernelGGL(k_colsum, dim3((27 * cout + 15) / 16), dim3(256), 0, (hipStream_t)stream,
                           (const float *)part, dw, grid, 27 * cout);
    } else {
        hipLaunchKernelGGL(k_conv3_small_wgrad, dim3(27 * cin * cout), dim3(256), 0, (hipStream_t)stream, in, dout, dw,
                           nx, ny, nz, cin, cout);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

long long ngapnet_small_wgrad_part_size(int cout) { return (long long)SW_BLOCKS * 27 * cout; }

int ngapnet_relu_bwd(const float *dy, const void *y, float *dx, void *dxb, long long n, void *stream) {
    const bool v4 = n % 4 == 0 && ((uintptr_t)dy | (uintptr_t)dx) % 16 == 0 && ((uintptr_t)y | (uintptr_t)dxb) % 8 == 0;
    if (v4)
        hipLaunchKernelGGL(k_relu_bwd_v4, dim3(blocks_for(n / 4)), dim3(256), 0, (hipStream_t)stream, dy,
                           (const __bf16 *)y, dx, (__bf16 *)dxb, n / 4);
    else
        hipLaunchKernelGGL(k_relu_bwd, dim3(blocks_for(n)), dim3(256), 0, (hipStream_t)stream, dy, (const __bf16 *)y,
                           dx, (__bf16 *)dxb, n);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_to_bf16(const float *s, void *d, long long n, void *stream) {
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks_for(n)), dim3(256), 0, (hipStream_t)stream, s, (__bf16 *)d, n);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_pool2(const void *in, void *out, int nx, int ny, int nz, int c, void *stream) {
    const long long n = (long long)nx * ny * nz * c / 8;
    if (c % 8 == 0 && ((uintptr_t)in | (uintptr_t)out) % 16 == 0)
        hipLaunchKernelGGL(k_pool2_v8, dim3(blocks_for(n / 8)), dim3(256), 0, (hipStream_t)stream, (const __bf16 *)in,
                           (__bf16 *)out, (__bf16 *)nullptr, nx, ny, nz, c, 0, 0);
    else
        hipLaunchKernelGGL(k_pool2, dim3(blocks_for(n)), dim3(256), 0, (hipStream_t)stream, (const __bf16 *)in,
                           (__bf16 *)out, nx, ny, nz, c);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_pool2_cat(const void *in, void *out, void *cat, int nx, int ny, int nz, int c, int ctot, int d0,
                      void *stream) {
    if (c % 8 == 0 && ctot % 8 == 0 && d0 % 8 == 0 && ((nx | ny | nz) & 1) == 0 &&
        ((uintptr_t)in | (uintptr_t)out | (uintptr_t)cat) % 16 == 0) {
        hipLaunchKernelGGL(k_pool2_v8, dim3(blocks_for((long long)nx * ny * nz * c / 64)), dim3(256), 0,
                           (hipStream_t)stream, (const __bf16 *)in, (__bf16 *)out, (__bf16 *)cat, nx, ny, nz, c, ctot, d0);
        return hipGetLastError() == hipSuccess ? 0 : 1;
    }
    const int rc = ngapnet_pool2(in, out, nx, ny, nz, c, stream);
    return rc ? rc : ngapnet_chan_copy_bf16(in, cat, (long long)nx * ny * nz, c, c, 0, ctot, d0, stream);
}

int ngapnet_pool2_bwd(const float *dout, float *din, int nx, int ny, int nz, int c, int acc, void *stream) {
    if (c % 4 == 0 && ((uintptr_t)dout | (uintptr_t)din) % 16 == 0)
        hipLaunchKernelGGL(k_pool2_bwd_v4, dim3(blocks_for((long long)nx * ny * nz * c / 4)), dim3(256), 0,
                           (hipStream_t)stream, dout, din, nx, ny, nz, c, acc);
    else
        hipLaunchKernelGGL(k_pool2_bwd, dim3(blocks_for((long long)nx * ny * nz * c)), dim3(256), 0,
                           (hipStream_t)stream, dout, din, nx, ny, nz, c, acc);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_up2(const void *in, void *out, int nx, int ny, int nz, int c, int ctot, int c0, void *stream) {
    if (c % 8 == 0 && ctot % 8 == 0 && c0 % 8 == 0 && ((uintptr_t)in | (uintptr_t)out) % 16 == 0)
        hipLaunchKernelGGL(k_up2_v8, dim3(blocks_for((long long)nx * ny * nz * c / 8)), dim3(256), 0,
                           (hipStream_t)stream, (const __bf16 *)in, (__bf16 *)out, nx, ny, nz, c, ctot, c0);
    else
        hipLaunchKernelGGL(k_up2, dim3(blocks_for((long long)nx * ny * nz * c)), dim3(256), 0, (hipStream_t)stream,
                           (const __bf16 *)in, (__bf16 *)out, nx, ny, nz, c, ctot, c0);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_up2_bwd(const float *dout, float *din, int nx, int ny, int nz, int c, int ctot, int c0, void *stream) {
    if (c % 4 == 0 && ctot % 4 == 0 && c0 % 4 == 0 && ((uintptr_t)dout | (uintptr_t)din) % 16 == 0)
        hipLaunchKernelGGL(k_up2_bwd_v4, dim3(blocks_for((long long)nx * ny * nz * c / 32)), dim3(256), 0,
                           (hipStream_t)stream, dout, din, nx, ny, nz, c, ctot, c0);
    else
        hipLaunchKernelGGL(k_up2_bwd, dim3(blocks_for((long long)nx * ny * nz * c / 8)), dim3(256), 0,
                           (hipStream_t)stream, dout, din, nx, ny, nz, c, ctot, c0);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_chan_copy_bf16(const void *src, void *dst, long long nv, int c, int cs, int s0, int cd, int d0,
                           void *stream) {
    return chan_copy((const __bf16 *)src, (__bf16 *)dst, nv, c, cs, s0, cd, d0, stream);
}

int ngapnet_chan_copy_f32(const float *src, float *dst, long long nv, int c, int cs, int s0, int cd, int d0,
                          void *stream) {
    return chan_copy(src, dst, nv, c, cs, s0, cd, d0, stream);
}

int ngapnet_conv1_fwd(const void *x, const float *w, float *y, long long nv, int c, void *stream) {
    if (c == 32)
        hipLaunchKernelGGL(k_conv1_fwd_t<32>, dim3(blocks_for(nv)), dim3(256), 0, (hipStream_t)stream,
                           (const __bf16 *)x, w, y, nv);
    else
        hipLaunchKernelGGL(k_conv1_fwd, dim3(blocks_for(nv)), dim3(256), 0, (hipStream_t)stream, (const __bf16 *)x, w,
                           y, nv, c);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_conv1_bwd(const void *x, const float *w, const float *dy, float *dx, float *dw, float *part, long long nv,
                      int c, void *stream) {
    if (c > 64) return -1;
    const int nb = 1024;
    if (c == 32)
        hipLaunchKernelGGL(k_conv1_bwd_t<32>, dim3(nb), dim3(256), 0, (hipStream_t)stream, (const __bf16 *)x, w, dy, dx,
                           part, nv);
    else
        hipLaunchKernelGGL(k_conv1_bwd, dim3(nb), dim3(256), 0, (hipStream_t)stream, (const __bf16 *)x, w, dy, dx,
                           part, nv, c);
    hipLaunchKernelGGL(k_colsum, dim3((c + 15) / 16), dim3(256), 0, (hipStream_t)stream, (const float *)part, dw, nb,
                       c);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_adam(float *w, const float *g, float *m, float *v, void *wb, long long n, float lr, float b1, float b2,
                 float eps, int step, float scale, void *stream) {
    float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(n)), dim3(256), 0, (hipStream_t)stream, w, g, m, v, (__bf16 *)wb, n, lr,
                       b1, b2, eps, c1, c2, scale);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ngapnet_sync(void) { return hipDeviceSynchronize() == hipSuccess ? 0 : 1; }

}  // extern "C"
