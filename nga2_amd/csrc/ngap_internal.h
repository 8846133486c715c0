// Internal declarations shared by the solver's translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "ngap_kernels.h"
#include "ngapsolve.h"

namespace ngap {

int grid_for(long long n);
int grid_parts(long long n);

template <typename T>
void launch_apply(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *x, T *y,
                  double *part);
// y = A x with the FP64 operator and x stored in FP32 (the mixed solve's
// search directions); part as in launch_apply
void launch_apply_x32(hipStream_t s, const Geo &g, const double *c, const double *a0, const double *a1,
                      const double *a2, const float *x, double *y, double *part);
// one symmetric-order Gauss-Seidel sweep, out of place (vin == nullptr: zero
// initial iterate); c1 = colour updated first (0 red, 1 black). Levels of rows
// <= 128 cells run whole-row tiles (k_sweep_row) unless tiles is set.
template <typename T>
void launch_sweep(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f,
                  const T *vin, T *vout, int c1, bool tiles = false);
// three transfers in one launch between level g[0] and g[3] (weights pm, pp of
// levels 1..3) along the directions dirs[0..2], whose chain_order is not 0
inline int chain_order(const int *dirs) {  // 0 unless the three differ
    return dirs[0] != dirs[1] && dirs[0] != dirs[2] && dirs[1] != dirs[2] ? 3 * dirs[0] + dirs[1] : 0;
}
template <typename T>
void launch_gather3(hipStream_t s, const Geo *g, int order, const T *const *pm, const T *const *pp, const T *r, T *fc);
template <typename T>
void launch_prolong3(hipStream_t s, const Geo *g, int order, const T *const *pm, const T *const *pp, const T *vc,
                     const T *vin, T *vout);
// true where launch_sweep2 takes k_sweep2_pair: FP32, even row length (x pairs),
// and no periodic direction of one cell in y or z (other periodic counts are even
// on every level; k_sweep2_pair colours by the unwrapped index). Offsets in a
// plane are 32 bits of bytes. And enough planes: a workgroup does at least 12
// steps for up to 6 planes, so on few planes the kernel is the better one only
// while its tiles run in few rounds on 256 CUs. Post- and pre-smoothing pair
// together against four single sweeps, us: 1024^2 x 1 110 and 70, x 2 110 and 89,
// x 3 112 and 107, x 4 114 and 124 (817 tiles); 720 x 728 x 2 58 and 59, x 3 58
// and 71 (403 tiles); 600 x 500 x 2 31 and 42 (231 tiles).
constexpr int PAIR_CX = 56, PAIR_CY = 24;  // output cells of its tiles
template <typename T>
inline bool pair_form(const Geo &g) {
    const long long tiles = (long long)((g.n0 + PAIR_CX - 1) / PAIR_CX) * ((g.n1 + PAIR_CY - 1) / PAIR_CY);
    return sizeof(T) == 4 && g.n0 % 2 == 0 && !(g.p1 && (g.n1 & 1)) && !(g.p2 && (g.n2 & 1)) &&
           (long long)g.n0 * g.n1 < (1LL << 30) && (g.n2 >= 4 || tiles <= 256LL * (g.n2 - 1));
}
// Levels whose sweeps run in fused pairs. With k_sweep2_pair from 2^19 cells on:
// 256^3 channel, FP32 V(2,2), 22.17 ms a solve with pairs on the fine level only,
// 21.05 from 2^23, 20.21 from 2^20, 20.10 from 2^19 and 2^18, 20.25 from 2^16
// (implicit 128^3: 5.17, 5.24, 4.90, 4.78, 4.84, 4.88 ms); below, a launch has too
// few planes per chunk and too few workgroups. With k_sweep2 on the largest levels
// only: at 256^3 the pair took 244 us against 2 x 131, and it was slower on the
// smaller ones.
template <typename T>
inline bool pairs_on(const Geo &g) {
    return g.N >= (pair_form<T>(g) ? 1LL << 19 : 1LL << 24);
}
// two fused sweeps of the same colour order (vin != vout); one_cell: the
// one-cell-per-lane kernel on every level
template <typename T>
void launch_sweep2(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f,
                   const T *vin, T *vout, int c1, bool one_cell = false);
// first symmetric sweep from a zero iterate as a stencil (no LDS)
template <typename T>
void launch_smooth0(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f, T *v,
                    int c1);
template <typename T>
void launch_resid(hipStream_t s, const Geo &g, const T *c, const T *a0, const T *a1, const T *a2, const T *f,
                  const T *x, T *r);
// fc = P^T r (vec = false: the one-cell-per-thread kernel on every level)
template <typename T>
void launch_gather(hipStream_t s, const Geo &F, const Geo &C, int d, const T *r, const T *pm, const T *pp, T *fc,
                   bool vec = true);
// vout = vin + P vc (vout may be vin; vin == nullptr: vout = P vc)
template <typename T>
void launch_prolong_to(hipStream_t s, const Geo &F, const Geo &C, int d, const T *pm, const T *pp, const T *vc,
                       const T *vin, T *vout, bool vec = true);
template <typename Tin, typename Tout>
void launch_dense(hipStream_t s, int n, const double *Ainv, const Tin *f, Tout *v);
int apply_blocks(const Geo &g, int &kc);

// The small levels of a V-cycle in one workgroup (see k_bottom).
constexpr int BOT_MAX_LEVELS = 16;
// Coarsening to the next level: the direction, and along it the cells and
// strides of this level and the next (all but d set by launch_bottom).
struct BotDir {
    int d, nf, nc, per, sf, sc;
};
template <typename T>
struct BotLevel {
    Geo g;
    BotDir dir;
    int relax;  // 0: skipped level (no smoothing, see set_relax)
    const T *c, *a0, *a1, *a2;
    const T *pm, *pp;  // transfer weights from the finer level (coarse-indexed)
    T *f, *v;
    float ih, i1;  // 1 / ceil(n0 / 2), 1 / n1 (set by launch_bottom)
};
template <typename T>
struct BotArgs {
    int nlev;  // levels lb..lb+nlev-1, the last one solved by the dense inverse
    int npre, npost;
    int cap;  // entries of the kernel's work arrays (set by launch_bottom)
    const double *Ainv;
    BotLevel<T> L[BOT_MAX_LEVELS];
};
// whether the n levels g[0] .. g[n-1] (the last the coarsest) fit the bottom kernel
template <typename T>
bool bottom_fits(const Geo *g, int n);
template <typename T>
void launch_bottom(hipStream_t s, const BotArgs<T> &a);
void launch_strength(hipStream_t s, const Geo &g, const double *a0, const double *a1, const double *a2, double *part,
                     int *nparts);
// counts of the cells with two or more directions and of the anisotropic ones
// (k_aniso_count) as block partials: part[0..nparts), part[MAX_PARTS..)
void launch_aniso_count(hipStream_t s, const Geo &g, const double *a0, const double *a1, const double *a2,
                        double *part, int *nparts);
// The coarsest level's dense (pseudo-)inverse in one workgroup (levels of at
// most COARSE_LDS_MAX cells): out[0] = 1 when singular, out[1] = 1 when the
// Cholesky factorisation failed.
constexpr int COARSE_LDS_MAX = 128;
void launch_coarse_inverse(hipStream_t s, const Geo &g, const double *c, const double *a0, const double *a1,
                           const double *a2, double *Ainv, double *out);
void launch_to_f32(hipStream_t s, long long n, const double *src, float *dst);
void launch_to_f64(hipStream_t s, long long n, const float *src, double *dst);

// One multigrid level on the device.
template <typename T>
struct LevelData {
    T *c = nullptr, *a0 = nullptr, *a1 = nullptr, *a2 = nullptr;
    T *pm = nullptr, *pp = nullptr; // weights of the transfer from the finer level (coarse-indexed)
    T *f = nullptr, *v = nullptr;   // right-hand side and final iterate (levels >= 1)
    T *w = nullptr;                 // second iterate buffer (out-of-place sweeps), all levels
};

// The coarse level's weights (pm, pp), couplings and diagonal from the fine
// level along direction d; with c32, their FP32 copies in the same pass.
void launch_coarse_build(hipStream_t s, const Geo &F, const Geo &C, int d, const double *c, const double *a0,
                         const double *a1, const double *a2, double *pm, double *pp, double *cc, double *ca0,
                         double *ca1, double *ca2, double *sc, const LevelData<float> *c32);

struct Level {
    Geo g{};
    int cdir = -1;
    bool relax = true;              // smoothed in the V-cycle (skipped relaxation)
    double str[3] = {0.0, 0.0, 0.0}; // sum |a_d| per direction, from the coarsening choice
    LevelData<double> d;
    LevelData<float> s;
};

}  // namespace ngap
