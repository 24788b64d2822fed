// Geometric multigrid V-cycle (the PCG preconditioner), red-black layout.
//
// Cell fields on smoothed levels are stored red-black compacted: plane c
// holds the cells of colour c = (x+y+z)&1 at (z, y, x>>1). A thread owns the
// x-pair (2m, 2m+1) of one row, i.e. compact index m in both planes, so every
// load is coalesced along m and a half-sweep touches only half of each field:
// one red-black Gauss-Seidel sweep reads r and z once and writes z once
// (3 field passes instead of 6 in the natural layout).
//
// Smoother: pre = (red, black)^nu from z = 0, post = (black, red)^nu (the
// adjoint order), R = P^T / 2^D with P separable cell-centred linear
// interpolation, coarsest level solved exactly by fast diagonalisation
// (tensor-product eigenbasis of the 1D operators) in FP64: the V-cycle is a
// symmetric positive definite preconditioner for CG.
#include <cmath>
#include <cstring>
#include <type_traits>
#include <utility>

#include "mg.hpp"
#include "mg_device.hpp"
#include "mg_leg.hpp"
#include "mg_rr.hpp"
#include "mg_tb.hpp"

namespace pano {

// ---- single-grid kernels: tile decode + the shared per-element bodies -------------------

#define RUN_TILE(G, NZ)                \
    int m, y, zb, L;                   \
    tile_xyz(G, m, y, zb, L);          \
    const int z0 = zb * (NZ);

// Red cells of the first sweep from z = 0 (the black half-sweep follows).
template <typename T, int DIM, int NZ>
__global__ __launch_bounds__(256) void k_red_init(Dims D, Grid3 G, T* zv, const T* r, T s, RInv<T> ri,
                                                  const SolverState* st) {
    if (st->done) return;
    RUN_TILE(G, NZ);
    if (m >= (D.w >> 1) || y >= D.h) return;
    red_init_run<T, DIM, NZ>(D, zv, r, s, ri, m, y, z0);
}

// The whole first sweep from z = 0 (2D levels: one launch instead of two).
template <typename T, int DIM, int NZ>
__global__ __launch_bounds__(256) void k_smooth_first(Dims D, Grid3 G, T* zv, const T* r, T s, RInv<T> ri,
                                                      const SolverState* st) {
    if (st->done) return;
    RUN_TILE(G, NZ);
    if (m >= (D.w >> 1) || y >= D.h) return;
    smooth_first_run<T, DIM, NZ>(D, zv, r, s, ri, m, y, z0);
}

// One colour of a red-black Gauss-Seidel sweep. With part, also the
// workgroup's partial sum of z.r over the updated cells.
template <typename T, int DIM, int NZ>
__global__ __launch_bounds__(256) void k_smooth_half(Dims D, Grid3 G, T* zv, const T* r, T s, RInv<T> ri,
                                                     int color, double* part, const SolverState* st) {
    if (st->done) return;
    RUN_TILE(G, NZ);
    double acc = 0.0;
    if (m < (D.w >> 1) && y < D.h) acc = smooth_half_run<T, DIM, NZ>(D, zv, r, s, ri, color, m, y, z0);
    if (part) {  // uniform across the workgroup
        double t = block_sum(acc);
        if (threadIdx.x == 0 && threadIdx.y == 0) part[L] = t;
    }
}

// res = r - s*(nc*z - sum)
template <typename T, int DIM, int NZ>
__global__ __launch_bounds__(256) void k_mg_residual(Dims D, Grid3 G, T* res, const T* zv, const T* r, T s,
                                                     const SolverState* st) {
    if (st->done) return;
    RUN_TILE(G, NZ);
    if (m >= (D.w >> 1) || y >= D.h) return;
    residual_run<T, DIM, NZ>(D, res, zv, r, s, m, y, z0);
}

// r_c = R res, NK coarse planes per thread
template <typename T, int DIM, int LC, int NK>
__global__ __launch_bounds__(256) void k_restrict(Dims Df, Dims Dc, Grid3 G, T* rc, const T* res,
                                                  const SolverState* st) {
    if (st->done) return;
    int I, J, kb, L;
    tile_xyz(G, I, J, kb, L);
    if (I >= Dc.w || J >= Dc.h) return;
    restrict_run<T, DIM, LC, NK>(Df, Dc, rc, res, I, J, kb * NK);
}

// z_o = z_f + P z_c (z_o may be z_f)
template <typename T, int DIM, int LC, int NZ>
__global__ __launch_bounds__(256) void k_prolong(Dims Df, Dims Dc, Grid3 G, T* zo, const T* zf, const T* zc,
                                                 const SolverState* st) {
    if (st->done) return;
    RUN_TILE(G, NZ);
    if (m >= (Df.w >> 1) || y >= Df.h) return;
    prolong_run<T, DIM, LC, NZ>(Df, Dc, zo, zf, zc, m, y, z0);
}

// ---- 3D f32 levels: prolongation from LDS ------------------------------------------------
// z_o = z_f + P z_c (3D; z_o may be z_f) on the pair tiles of grid3_rb, with
// the workgroup's coarse neighbourhood ((kTX+2) x (kTY/2+2) x ((NZ+1)/2+2)
// cells) copied to LDS first; the arithmetic of prolong_run.
template <int LC, int NZ>
__global__ __launch_bounds__(256) void k_prolong3_lds(Dims Df, Dims Dc, Grid3 G, float* zo, const float* zf,
                                                      const float* zc, const SolverState* st) {
    if (st->done) return;
    constexpr int CX = kTX + 2, CY = kTY / 2 + 2, CZ = (NZ + 1) / 2 + 2;
    __shared__ float ct[CZ * CY * CX];
    const int L = xcd_remap(blockIdx.x, G.nb);
    const int bx = L % G.gx, tq = L / G.gx, by = tq % G.gy, bz = tq / G.gy;
    const int m0 = bx * kTX, y0 = by * kTY, z0 = bz * NZ;
    const int Ib = m0 - 1, Jb = (y0 >> 1) - 1, Kb = (z0 >> 1) - 1;
    const int tid = threadIdx.x + kTX * threadIdx.y;
    constexpr int NP = (CZ * CY * CX + kTX * kTY - 1) / (kTX * kTY);
    float vc[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {  // all loads first (clamped, valid indices)
        int e = imin(tid + i * kTX * kTY, CZ * CY * CX - 1);
        int ix = e % CX, t2 = e / CX, iy = t2 % CY, iz = t2 / CY;
        int I = imin(imax(Ib + ix, 0), Dc.w - 1);
        int J = imin(imax(Jb + iy, 0), Dc.h - 1);
        int K = imin(imax(Kb + iz, 0), Dc.d - 1);
        vc[i] = ldx(zc, cidx<LC>(Dc, K, J, I));
    }
    // the thread's fine values too, before the barrier (clamped to a valid cell
    // for threads past the grid's edge, which store nothing)
    const int m = m0 + threadIdx.x, y = y0 + threadIdx.y;
    const bool mine = m < (Df.w >> 1) && y < Df.h;
    float f0[NZ], f1[NZ];
    int i0[NZ], i1[NZ];
#pragma unroll
    for (int k = 0; k < NZ; ++k) {
        RBRow R = rb_row<3>(Df, zclamp(Df, z0 + k), mine ? y : 0, mine ? m : 0);
        i0[k] = R.i0;
        i1[k] = R.i1;
        f0[k] = ldx(zf, R.i0);
        f1[k] = ldx(zf, R.i1);
    }
#pragma unroll
    for (int i = 0; i < NP; ++i)
        if (tid + i * kTX * kTY < CZ * CY * CX) ct[tid + i * kTX * kTY] = vc[i];
    __syncthreads();
    if (!mine) return;
    const float w34 = 0.75f, w14 = 0.25f, one = 1.0f, zero = 0.0f;
    int J0, J1;
    bool ey;
    p1(y, Dc.h, J0, J1, ey);
    const float wy0 = ey ? one : w34, wy1 = ey ? zero : w14;
    const bool el = m == 0, er = m + 1 >= Dc.w;
    const int Il = el ? m : m - 1, Ir = er ? m : m + 1;
    const float wl0 = el ? one : w34, wl1 = el ? zero : w14;
    const float wr0 = er ? one : w34, wr1 = er ? zero : w14;
#pragma unroll
    for (int k = 0; k < NZ; ++k) {
        int z = z0 + k;
        if (z >= Df.d) continue;
        int K0, K1;
        bool ez;
        p1(z, Dc.d, K0, K1, ez);
        const float wz0 = ez ? one : w34, wz1 = ez ? zero : w14;
        float px0[2][2], px1[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const float* row = ct + (((a == 0 ? K0 : K1) - Kb) * CY + ((b == 0 ? J0 : J1) - Jb)) * CX - Ib;
                float cm = row[m], cl = row[Il], cr = row[Ir];
                px0[a][b] = wl0 * cm + wl1 * cl;
                px1[a][b] = wr0 * cm + wr1 * cr;
            }
        float v0 = wz0 * (wy0 * px0[0][0] + wy1 * px0[0][1]) + wz1 * (wy0 * px0[1][0] + wy1 * px0[1][1]);
        float v1 = wz0 * (wy0 * px1[0][0] + wy1 * px1[0][1]) + wz1 * (wy0 * px1[1][0] + wy1 * px1[1][1]);
        stx(zo, i0[k], f0[k] + v0);
        stx(zo, i1[k], f1[k] + v1);
    }
}

// ---- 3D f32 levels: the pre- and post-smoothing as one pass each ----------------------
// NS half-sweeps from xin into xout (TbThread); with DOT the workgroup's sums
// of z.r over its tile for the last two half-sweeps go to part[L] and
// part[nb + L]. PL >= 0: from xin + P zco (zco: the coarse level, layout PL,
// dims Dc) instead of xin.
template <int TXP, int TY, int NT, int WPE, int CF, bool ZERO_X, bool DOT, int PL>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE))) void k_smooth_tb(
    Dims D, TbGrid g, const float* xin, float* xout, const float* r, float s, RInv<float> ri, double* part,
    const float* zco, Dims Dc, const SolverState* st) {
    if (st->done) return;
    __shared__ float lds[TbThread<4, TXP, TY, NT, CF, ZERO_X, DOT, PL>::LDS_FLOATS];
    const int L = xcd_remap(blockIdx.x, g.nb);
    const int bx = L % g.gx, q = L / g.gx, by = q % g.gy, bz = q / g.gy;
    double acc[2];
    tb_workgroup<TXP, TY, NT, CF, ZERO_X, DOT, PL>(lds, D, bx, by, bz, g.zc, xin, xout, r, s, ri.v, acc, zco, Dc);
    if constexpr (DOT) {
        double a0 = acc[0], a1 = acc[1];
        block_sum2<NT>(a0, a1);
        if (threadIdx.x == 0) {
            part[L] = a0;
            part[g.nb + L] = a1;
        }
    }
}

// The 2D form: one workgroup per tile of a 2D level.
template <int TXP, int TY, int NT, int WPE, int CF, bool ZERO_X, bool DOT, int PL>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE))) void k_smooth_tb2(
    Dims D, TbGrid g, const float* xin, float* xout, const float* r, float s, RInv<float> ri, double* part,
    const float* zco, Dims Dc, const SolverState* st) {
    if (st->done) return;
    __shared__ float lds[Tb2Thread<4, TXP, TY, NT, CF, ZERO_X, DOT, PL>::LDS_FLOATS];
    const int L = xcd_remap(blockIdx.x, g.nb);
    const int bx = L % g.gx, by = L / g.gx;
    double acc[2];
    tb2_workgroup<TXP, TY, NT, CF, ZERO_X, DOT, PL>(lds, D, bx, by, xin, xout, r, s, ri.v, acc, zco, Dc);
    if constexpr (DOT) {
        double a0 = acc[0], a1 = acc[1];
        block_sum2<NT>(a0, a1);
        if (threadIdx.x == 0) {
            part[L] = a0;
            part[g.nb + L] = a1;
        }
    }
}

// The four half-sweeps (colours CF, CF^1, ...) of a 3D f32 level in one pass;
// with part, the z.r partials (2 per workgroup, *np set). PL >= 0: the
// sweeps start from xin + P zco, zco the coarse level (layout PL, dims Dc).
template <int CF, bool ZERO_X, bool DOT, int PL = -1>
static void smooth_tb(Ctx* c, const char* name, double bytes, const Dims& D, const float* xin, float* xout,
                      const float* r, float s, const RInv<float>& ri, double* part, int* np, const SolverState* st,
                      const float* zco = nullptr, const Dims& Dc = Dims{}) {
    if (D.d <= 1) {
        using C = Tb2D;
        const TbGrid g = tb2_grid(D);
        klaunch(c, name, bytes, k_smooth_tb2<C::TXP, C::TY, C::NT, C::WPE, CF, ZERO_X, DOT, PL>, dim3(g.nb),
                dim3(C::NT), D, g, xin, xout, r, s, ri, part, zco, Dc, st);
        if (np) *np = 2 * g.nb;
        return;
    }
    with_tb(D, [&](auto cfg) {
        using C = decltype(cfg);
        const TbGrid g = tb_grid_of<C>(D);
        klaunch(c, name, bytes, k_smooth_tb<C::TXP, C::TY, C::NT, C::WPE, CF, ZERO_X, DOT, PL>, dim3(g.nb),
                dim3(C::NT), D, g, xin, xout, r, s, ri, part, zco, Dc, st);
        if (np) *np = 2 * g.nb;
        return 0;
    });
}

// Tile shape, plane chunks and load-ahead depth of the one-pass residual +
// restriction. It streams plane by plane, so a workgroup's time is a chain of
// load latencies: on levels below 2^23 cells the two separate kernels (more
// workgroups, no chain) are faster.
constexpr int kRrWant = 512, kRrKmin = 2, kRrPD = 1;
// Its tiles, coarse cells in x by rows, 512 threads and two workgroups per CU
// each. A tile's rows are read with two pairs more on each side, which are two
// more 128-byte lines per colour, so its L2 misses fall with its width: at 512^3
// 32 x 8 tiles fetched 2.1 times the field and ran at the memory's rate.
// Level 0 of 512^3 / 256^3, us: 32 x 8 381 / 42, 32 x 16 343 / 36, 64 x 8
// 304 / 35, 64 x 16 (one workgroup per CU) 304 / 36, 64 x 4 341 / 43; twice
// the workgroups in shorter chunks 295 / 41. Wide tiles, unless the level's
// edges leave them more than a tenth more padded cells than narrow ones.
constexpr int kRrWideX = 64, kRrWideY = 8, kRrNarrowX = 32, kRrNarrowY = 16;
inline bool rr_wide(const Dims& Dc) {
    auto padded = [&](int tx, int ty) { return (int64_t)((Dc.w + tx - 1) / tx * tx) * ((Dc.h + ty - 1) / ty * ty); };
    return 10 * padded(kRrWideX, kRrWideY) <= 11 * padded(kRrNarrowX, kRrNarrowY);
}
inline bool rr_on(bool enabled, const Dims& D) {
    return enabled && D.d > 1 && (int64_t)D.d * D.h * D.w >= (int64_t(1) << 23);
}

// r_c = R (r - A z) of a 3D f32 level in one pass (no fine residual in HBM).
template <int TXC, int TYC, int LC>
__global__ __launch_bounds__(TXC * TYC) void k_resrestrict(Dims D, Dims Dc, RrGrid g, const float* z, const float* b,
                                                           float* rc, float s, const SolverState* st) {
    if (st->done) return;
    __shared__ float lds[RrShape<TXC, TYC>::LDS_FLOATS];
    const int L = xcd_remap(blockIdx.x, g.nb);
    const int bx = L % g.gx, q = L / g.gx, by = q % g.gy, bz = q / g.gy;
    rr_workgroup<TXC, TYC, LC, kRrPD>(lds, D, Dc, bx, by, bz, g.kc, z, b, rc, s);
}

// The 2D form: one workgroup per tile of coarse cells, one plane.
template <int LC>
__global__ __launch_bounds__(kRr2TX * kRr2TY) void k_resrestrict2(Dims D, Dims Dc, int gx, int nb, const float* z,
                                                                  const float* b, float* rc, float s,
                                                                  const SolverState* st) {
    if (st->done) return;
    __shared__ float lds[Rr2Thread<kRr2TX, kRr2TY, LC>::LDS_FLOATS];
    const int L = xcd_remap(blockIdx.x, nb);
    rr2_workgroup<kRr2TX, kRr2TY, LC>(lds, D, Dc, L % gx, L / gx, z, b, rc, s);
}

template <int LC>
static void resrestrict2(Ctx* c, const char* name, double bytes, const Dims& D, const Dims& Dc, const float* z,
                         const float* b, float* rc, float s, const SolverState* st) {
    const int gx = (Dc.w + kRr2TX - 1) / kRr2TX, gy = (Dc.h + kRr2TY - 1) / kRr2TY;
    klaunch(c, name, bytes, k_resrestrict2<LC>, dim3(gx * gy), dim3(kRr2TX * kRr2TY), D, Dc, gx, gx * gy, z, b, rc,
            s, st);
}

template <int LC>
static void resrestrict(Ctx* c, const char* name, double bytes, const Dims& D, const Dims& Dc, const float* z,
                        const float* b, float* rc, float s, const SolverState* st) {
    auto launch = [&](auto kern, const RrGrid& g, int nt) {
        klaunch(c, name, bytes, kern, dim3(g.nb), dim3(nt), D, Dc, g, z, b, rc, s, st);
    };
    if (rr_wide(Dc))
        launch(k_resrestrict<kRrWideX, kRrWideY, LC>, rr_grid<kRrWideX, kRrWideY>(Dc, kRrWant, kRrKmin),
               kRrWideX * kRrWideY);
    else
        launch(k_resrestrict<kRrNarrowX, kRrNarrowY, LC>, rr_grid<kRrNarrowX, kRrNarrowY>(Dc, kRrWant, kRrKmin),
               kRrNarrowX * kRrNarrowY);
}

// ---- a level's legs as one launch each (mg_leg.hpp) ------------------------------------
// Tiles: 2D 32 x-pairs by 16 rows; 3D 8 x-pairs by 8 rows by 8 planes, or by 2
// planes where those are few enough to run at once (leg_thin: a workgroup's
// time grows with its planes: 32^3 8.0 / 8.2 us with 8 planes, 6.6 / 6.6 with
// 2; 64^3, 1024 workgroups with 2 planes, 9.8 / 9.2 against 17.0 / 15.6).
template <typename T, int DIM, bool DOWN, bool THIN>
using LegS = LegShape<T, DIM, DIM == 3 ? 8 : 32, DIM == 3 ? 8 : 16, DIM == 2 ? 1 : THIN ? 2 : 8, DOWN>;
inline bool leg_thin(const Dims& D) {
    return D.d > 1 && leg_grid<LegS<float, 3, true, true>>(D).nb <= 256;
}
// f(integral_constant<bool, THIN>) of a level
template <int DIM, class F>
inline void with_leg(const Dims& D, F&& f) {
    if constexpr (DIM == 3) {
        if (leg_thin(D)) return f(std::true_type{});
    }
    f(std::false_type{});
}

template <typename T, int DIM, bool THIN, int LC>
__global__ __launch_bounds__((LegS<T, DIM, true, THIN>::NT)) void k_leg_down(Dims D, Dims Dc, LegGrid g, T* zo, const T* r,
                                                                       T* rc, T s, RInv<T> ri, const SolverState* st) {
    if (st->done) return;
    using S = LegS<T, DIM, true, THIN>;
    __shared__ T lds[S::LDS / sizeof(T)];
    const int L = xcd_remap(blockIdx.x, g.nb);
    leg_down<T, DIM, S, LC>(lds, D, Dc, L % g.gx, L / g.gx % g.gy, L / (g.gx * g.gy), zo, r, rc, s, ri);
}

template <typename T, int DIM, bool THIN, int LC, bool DOT>
__global__ __launch_bounds__((LegS<T, DIM, false, THIN>::NT)) void k_leg_up(Dims D, Dims Dc, LegGrid g, const T* zd, T* zo,
                                                                      const T* r, const T* zc, T s, RInv<T> ri,
                                                                      double* part, const SolverState* st) {
    if (st->done) return;
    using S = LegS<T, DIM, false, THIN>;
    __shared__ T lds[S::LDS / sizeof(T)];
    const int L = xcd_remap(blockIdx.x, g.nb);
    double acc[2] = {0.0, 0.0};
    leg_up<T, DIM, S, LC, DOT>(lds, D, Dc, L % g.gx, L / g.gx % g.gy, L / (g.gx * g.gy), zd, zo, r, zc, s, ri, acc);
    if constexpr (DOT) {
        block_sum2<S::NT>(acc[0], acc[1]);
        if (threadIdx.x == 0) {
            part[L] = acc[0];
            part[g.nb + L] = acc[1];
        }
    }
}

// Whether level l runs its legs as one launch each: where the halo cells that
// every workgroup recomputes are cheaper than the launches. Against the
// separate kernels, 3D both legs: f32 64^3 19 against 30 us, 96^3 39 against
// 65, 128^3 about 85 against 45; f64 64^3 21 against 44, 96^3 55 against 65,
// 128^3 109 against 99. 2D down leg: f32 512^2 4.6 against 8.7 us, 1024^2 9.2
// against 10, 2048^2 30 against 26; f64 2048^2 36 against 66 (up 49 against 61).
template <typename T>
static bool leg_on(const MG<T>* m, int l) {
    const Dims& D = m->dims[l];
    const int64_t n = (int64_t)D.d * D.h * D.w, M = int64_t(1) << 20;
    if (!m->pro || !m->tb || m->nu != 2 || l + 1 >= m->levels) return false;
    if (D.d > 1) return n < M;
    return std::is_same<T, double>::value || n <= M;
}
// Up leg: f32 2D levels keep the one-pass smoother (32 x 32 tiles).
template <typename T>
static bool leg_up_on(const MG<T>* m, int l) {
    return leg_on(m, l) && (std::is_same<T, double>::value || m->dims[l].d > 1);
}

// ---- coarsest level: fast diagonalisation in FP64 (natural layout) ---------------------
// 1D operator along one axis with n cells: diag = (i>0 ? 1 : lo) + (i<n-1 ? 1 : hi),
// off-diagonal -1 (lo/hi = 1 for an open side). Closed-form eigenpairs:
//  wall/wall: cos(pi k (j+1/2)/n),            lambda = 2 - 2 cos(pi k/n)
//  wall/open: cos(pi (2k+1)(j+1/2)/(2n+1)),   lambda = 2 - 2 cos(pi (2k+1)/(2n+1))
//  open/wall: the mirror image of wall/open
//  open/open: sin(pi (k+1)(j+1)/(n+1)),       lambda = 2 - 2 cos(pi (k+1)/(n+1))
// Vectors normalised; the eigen-residual is checked in double.
static pano_status eig1d(int n, int lo, int hi, std::vector<double>& V, std::vector<double>& lam) {
    V.assign((size_t)n * n, 0.0);
    lam.assign(n, 0.0);
    const double pi = 3.14159265358979323846;
    for (int k = 0; k < n; ++k) {
        double theta;
        for (int j = 0; j < n; ++j) {
            double v;
            if (!lo && !hi) { theta = pi * k / n; v = std::cos(theta * (j + 0.5)); }
            else if (!lo && hi) { theta = pi * (2 * k + 1) / (2 * n + 1); v = std::cos(theta * (j + 0.5)); }
            else if (lo && !hi) { theta = pi * (2 * k + 1) / (2 * n + 1); v = std::cos(theta * ((n - 1 - j) + 0.5)); }
            else { theta = pi * (k + 1) / (n + 1); v = std::sin(theta * (j + 1)); }
            V[(size_t)j * n + k] = v;
        }
        if (!lo && !hi) theta = pi * k / n;
        else if (lo && hi) theta = pi * (k + 1) / (n + 1);
        else theta = pi * (2 * k + 1) / (2 * n + 1);
        lam[k] = 2.0 - 2.0 * std::cos(theta);
        double nn = 0.0;
        for (int j = 0; j < n; ++j) nn += V[(size_t)j * n + k] * V[(size_t)j * n + k];
        nn = std::sqrt(nn);
        for (int j = 0; j < n; ++j) V[(size_t)j * n + k] /= nn;
    }
    // residual check ||T v - lambda v||_inf
    double worst = 0.0;
    for (int k = 0; k < n; ++k)
        for (int j = 0; j < n; ++j) {
            double dg = (j > 0 ? 1.0 : lo) + (j < n - 1 ? 1.0 : hi);
            double tv = dg * V[(size_t)j * n + k];
            if (j > 0) tv -= V[(size_t)(j - 1) * n + k];
            if (j < n - 1) tv -= V[(size_t)(j + 1) * n + k];
            double e = std::fabs(tv - lam[k] * V[(size_t)j * n + k]);
            worst = e > worst ? e : worst;
        }
    if (worst > 1e-9) return fail(PANO_ERR_DEVICE, "eigen-basis check failed (n=%d, err=%g)", n, worst);
    return PANO_OK;
}

// Device copy of the eigenbasis of one axis, cached per (n, lo, hi): V, followed
// by its transpose (basis_t), which the matrix products read row by row where V
// would be read column by column.
pano_status axis_basis(Ctx* c, int n, int lo, int hi, double** V, double** lam) {
    char key[64];
    snprintf(key, sizeof(key), "eig:%d:%d:%d", n, lo, hi);
    auto it = c->consts.find(key);
    if (it == c->consts.end()) {
        std::vector<double> hv, hl;
        PANO_CHECK(eig1d(n, lo, hi, hv, hl));
        void* p = nullptr;
        const size_t nn = (size_t)n * n;
        std::vector<double> all(2 * nn + n);  // V, its transpose, the eigenvalues
        for (int j = 0; j < n; ++j)
            for (int k = 0; k < n; ++k) {
                all[(size_t)j * n + k] = hv[(size_t)j * n + k];
                all[nn + (size_t)k * n + j] = hv[(size_t)j * n + k];
            }
        std::copy(hl.begin(), hl.end(), all.begin() + 2 * nn);
        const size_t bytes = all.size() * sizeof(double);
        if (hipMalloc(&p, bytes) != hipSuccess) {
            (void)hipGetLastError();
            return fail(PANO_ERR_OOM, "eigenbasis allocation failed");
        }
        PANO_HIP(hipMemcpy(p, all.data(), bytes, hipMemcpyHostToDevice));
        it = c->consts.emplace(key, p).first;
    }
    *V = (double*)it->second;
    *lam = (double*)it->second + 2 * (size_t)n * n;
    return PANO_OK;
}

pano_status mg_check(const Dims& D, int levels) {
    if (levels < 2 || levels > 12) return fail(PANO_ERR_BAD_SHAPE, "mg_levels must be in [2, 12] (got %d)", levels);
    int f = 1 << (levels - 1);
    if (D.w % (2 * (f / 2 > 0 ? f / 2 : 1)) != 0 || D.w % f != 0 || D.h % f != 0 || (D.d > 1 && D.d % f != 0))
        return fail(PANO_ERR_BAD_SHAPE,
                    "multigrid with %d levels needs every extent divisible by %d (got %dx%dx%d)", levels, f, D.d,
                    D.h, D.w);
    // smoothed levels 0..levels-2 need an even x extent
    if (((D.w >> (levels - 2)) & 1) != 0)
        return fail(PANO_ERR_BAD_SHAPE, "multigrid needs an even x extent on every smoothed level");
    int cw = D.w >> (levels - 1), ch = D.h >> (levels - 1), cd = D.d > 1 ? D.d >> (levels - 1) : 1;
    if (cw > 256 || ch > 256 || cd > 256)
        return fail(PANO_ERR_BAD_SHAPE, "coarsest multigrid level %dx%dx%d too large (max 256 per axis); use more levels",
                    cd, ch, cw);
    if (cw < 1 || ch < 1 || cd < 1) return fail(PANO_ERR_BAD_SHAPE, "too many multigrid levels");
    return PANO_OK;
}

static bool fdm_split_on(const Dims& C);

// Level l (above the coarsest) of a 3D f32 hierarchy runs its prolongation
// inside the one-pass post-smoothing.
template <typename T>
static bool pro_level(const MG<T>* m, int l) {
    return m->pro && l + 1 < m->levels &&
           ((std::is_same<T, float>::value && tb_on(m->tb, m->nu, m->dims[l])) || leg_on(m, l));
}

template <typename T>
pano_status mg_setup(Ctx* c, const Dims& D, int levels, int nu, double dt, MG<T>* m) {
    PANO_CHECK(mg_check(D, levels));
    m->levels = levels;
    m->nu = nu;
    const char* fused = getenv("PANO_MG_FUSED");
    m->tb = !(fused && fused[0] == '0');
    double s = dt;
    for (int l = 0; l < levels; ++l) {
        Dims Dl = D;
        Dl.w = D.w >> l;
        Dl.h = D.h >> l;
        Dl.d = D.d > 1 ? D.d >> l : 1;
        m->dims[l] = Dl;
        m->s[l] = s;
        s *= 0.25;
        if (l >= 1) {
            int64_t n = (int64_t)Dl.d * Dl.h * Dl.w;
            char kz[32], kr[32];
            snprintf(kz, sizeof(kz), "mg_z%d", l);
            snprintf(kr, sizeof(kr), "mg_r%d", l);
            void* pz;
            void* pr;
            PANO_CHECK(c->workspace(kz, n * sizeof(T), &pz));
            PANO_CHECK(c->workspace(kr, n * sizeof(T), &pr));
            m->z[l] = (T*)pz;
            m->r[l] = (T*)pr;
        }
    }
    const char* pro = getenv("PANO_MG_PRO");
    m->pro = !(pro && pro[0] == '0');
    for (int l = 0; l + 1 < levels; ++l) {
        m->w[l] = nullptr;
        if (!pro_level(m, l)) continue;
        const Dims& Dl = m->dims[l];
        char kw[32];
        snprintf(kw, sizeof(kw), "mg_w%d", l);
        void* pw;
        PANO_CHECK(c->workspace(kw, (size_t)Dl.d * Dl.h * Dl.w * sizeof(T), &pw));
        m->w[l] = (T*)pw;
    }
    void* pres;
    PANO_CHECK(c->workspace("mg_res", (size_t)D.d * D.h * D.w * sizeof(T), &pres));
    m->res = (T*)pres;
    const Dims& C = m->dims[levels - 1];
    int64_t nc = (int64_t)C.d * C.h * C.w;
    void* t0;
    void* t1;
    PANO_CHECK(c->workspace("fdm_t0", nc * sizeof(double), &t0));
    PANO_CHECK(c->workspace("fdm_t1", nc * sizeof(double), &t1));
    m->fdm_tmp[0] = (double*)t0;
    m->fdm_tmp[1] = (double*)t1;
    m->coarse_n[0] = C.w;
    m->coarse_n[1] = C.h;
    m->coarse_n[2] = C.d;
    m->fdm_split = fdm_split_on(C);
    PANO_CHECK(axis_basis(c, C.w, C.bc & 1, (C.bc >> 1) & 1, &m->fdm_v[0], &m->fdm_lam[0]));
    PANO_CHECK(axis_basis(c, C.h, (C.bc >> 2) & 1, (C.bc >> 3) & 1, &m->fdm_v[1], &m->fdm_lam[1]));
    // a 3D hierarchy may end in a single plane, which its z pass still transforms
    if (D.d > 1) PANO_CHECK(axis_basis(c, C.d, (C.bc >> 4) & 1, (C.bc >> 5) & 1, &m->fdm_v[2], &m->fdm_lam[2]));
    else { m->fdm_v[2] = nullptr; m->fdm_lam[2] = nullptr; }
    return PANO_OK;
}

// ---- coarsest level in LDS ---------------------------------------------------------------
// One workgroup per plane (per y-row for the z pass): 1024 threads, so the
// LDS-latency-bound dot products of a slice have 4 waves per SIMD to overlap.
constexpr int kFdmThreads = 1024;
template <typename Tin, typename Tout>
__global__ __launch_bounds__(kFdmThreads) void k_fdm_plane(int nx, int ny, int mode, const Tin* in, Tout* out,
                                                   const double* Vx, const double* Vy, const double* lx,
                                                   const double* ly, double s, double eps,
                                                   const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    int64_t P = (int64_t)nx * ny;
    fdm_plane_body<Tin, Tout>(fdm_lds, nx, ny, mode, in + blockIdx.x * P, out + blockIdx.x * P, Vx, Vy, lx, ly, s,
                              eps);
}

// The first pass of the 3D coarsest solve with its right-hand side restricted
// from the fine residual (red-black layout, level dims Df) on the fly:
// plane K's element (J, I) is restrict_value3, the value k_restrict stores,
// so the coarse right-hand side is never written.
__global__ __launch_bounds__(kFdmThreads) void k_fdm_plane_rc(Dims Df, Dims Dc, const float* res, double* out,
                                                      const double* Vx, const double* Vy, double s, double eps,
                                                      const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    const int nx = Dc.w, ny = Dc.h, K = blockIdx.x;
    fdm_plane_body_src<double>(
        fdm_lds, nx, ny, 0,
        [&](int e) {
            const int J = e / nx, I = e - J * nx;
            return (double)restrict_value3<float>(Df, Dc, res, I, J, K);
        },
        out + (int64_t)K * nx * ny, Vx, Vy, (const double*)nullptr, (const double*)nullptr, s, eps);
}

template <typename Tin, typename Tout>
__global__ __launch_bounds__(256) void k_fdm2_tile(int nx, int ny, int pass, const Tin* in, Tout* out,
                                                   const double* Vx, const double* Vy, const double* lx,
                                                   const double* ly, double s, double eps, const SolverState* st) {
    if (st->done) return;
    __shared__ double lds[1024];
    fdm2_tile_body<Tin, Tout>(lds, nx, ny, blockIdx.x, pass, in, out, Vx, Vy, lx, ly, s, eps);
}

template <typename T>
__global__ __launch_bounds__(kFdm2Threads) void k_fdm2_one(int nx, int ny, const T* in, T* out, const double* Vx,
                                                           const double* Vy, const double* lx, const double* ly,
                                                           double s, double eps, const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    fdm2_one_body<T, T>(fdm_lds, nx, ny, in, out, Vx, Vy, lx, ly, s, eps);
}

__global__ __launch_bounds__(kFdmThreads) void k_fdm_zcol(int nx, int ny, int nz, double* data, const double* Vz,
                                                  const double* lx, const double* ly, const double* lz, double s,
                                                  double eps, const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    fdm_zcol_body(fdm_lds, nx, ny, nz, blockIdx.x, data, Vz, lx, ly, lz, s, eps);
}

// ---- 3D coarsest level: FP64 matrix products on the matrix cores -----------------------
// The six products of the solve, x, y, z forward, the division, z, y, x inverse,
// in 16 x 16 tiles of v_mfma_f64_16x16x4 (mfma_tile). Every output is the same
// chain of fused multiply-adds in the same order (q = 0 .. n-1 from 0) as
// lds_axis's, so the results are those of k_fdm_plane / k_fdm_zcol bit for bit.
// With a sum per thread, two LDS reads per product bounded the passes.
//
// Three launches for any size, each two products with the first one's result
// in LDS, split over the index both leave free (64^3: 256 workgroups each):
//  forward: plane K, 16 columns i: x for them (every row), then y;
//  z:       16 cells of a plane: z forward, divide, z inverse;
//  inverse: plane K, 16 rows j: y for them (every column), then x.
// 64^3 53 + 28 + 49 us with a sum per thread, 7 + 7 + 9 now; 32^3 6.4 + 5.8 +
// 5.4, now 4.6 + 4.6 + 4.8 (launch and two rounds of loads).
// An axis past 64 cells has 16 waves per workgroup instead of four, a tile each;
// and where that leaves few workgroups their long products are split, or one
// workgroup's CU reads the whole basis: y forward below 64 workgroups, z up to
// 128. Two-level V-cycles, us, with a sum per thread / four waves / now: coarsest
// level 256 x 8 x 8 (z, y, x) 75 / 91 / 55, 8 x 256 x 8 69 / 81 / 58, 7 x 4 x 248
// 56 / 59 / 53, 256 x 32 x 32 263 / 135 / 93, 128^3 2147 / 380 / 339. (256 x 48 x
// 48, 144 workgroups in z: 157 not split, 154 split, f64 215 and 221.)
__device__ __forceinline__ const double* basis_t(const double* V, int n) { return V + (size_t)n * n; }
constexpr int kFdm3P = 17;  // row length in LDS of a block of 16 columns
inline size_t fdm3_lds_cols(int n) { return (size_t)((n + 15) / 16 * 16) * kFdm3P * sizeof(double); }
__host__ __device__ inline int fdm3_row(int nx) { return (nx + 15) / 16 * 16 + 2; }

// forward x then y of plane K, columns [i0, i0 + 16): in -> out (double); the
// rows of y, with the whole x product before them, may be split over gridDim.y
template <typename Tin, int NT>
__global__ __launch_bounds__(NT) void k_fdm3_fwd(int nx, int ny, const Tin* in, double* out, const double* Vx,
                                                 const double* Vy, const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    const int gx = (nx + 15) >> 4, K = blockIdx.x / gx, i0 = (blockIdx.x - K * gx) * 16;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, h = lane >> 4, gy = (ny + 15) >> 4;
    const int ic = imin(i0 + r, nx - 1);
    const Tin* src = in + (int64_t)K * nx * ny;
    double* dst = out + (int64_t)K * nx * ny;
    for (int jt = w; jt < gy; jt += NT / 64) {
        const int jc = imin(jt * 16 + r, ny - 1);
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
        mfma_tile<8>(0, nx, [&](int q) { return (double)src[jc * nx + q]; }, [&](int q) { return Vx[q * nx + ic]; },
                     acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) fdm_lds[(jt * 16 + 4 * v + h) * kFdm3P + r] = acc[v];
    }
    __syncthreads();
    const int jn = (gy + gridDim.y - 1) / gridDim.y, j0 = blockIdx.y * jn, j1 = imin(j0 + jn, gy);
    for (int jt = j0 + w; jt < j1; jt += NT / 64) {
        const int jc = imin(jt * 16 + r, ny - 1);
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
        mfma_tile<8>(0, ny, [&](int q) { return Vy[q * ny + jc]; }, [&](int q) { return fdm_lds[q * kFdm3P + r]; },
                     acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = jt * 16 + 4 * v + h;
            if (j < ny && i0 + r < nx) dst[j * nx + i0 + r] = acc[v];
        }
    }
}

// cells [e0, e0 + 16) of every plane: z forward, divide by s*(lx+ly+lz) (0 on
// the null space), z inverse, in place on data (double)
template <int NT>
__global__ __launch_bounds__(NT) void k_fdm3_z(int nx, int ny, int nz, double* data, const double* Vz,
                                               const double* lx, const double* ly, const double* lz, double s,
                                               double eps, const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    const int P = nx * ny, lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, h = lane >> 4;
    const int e = blockIdx.x * 16 + r, ec = imin(e, P - 1), gz = (nz + 15) >> 4;
    const double lxy = lx[ec % nx] + ly[ec / nx];
    const double* Wz = basis_t(Vz, nz);
    for (int kt = w; kt < gz; kt += NT / 64) {
        const int kc = imin(kt * 16 + r, nz - 1);
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
        mfma_tile<8>(0, nz, [&](int q) { return Vz[q * nz + kc]; }, [&](int q) { return data[(int64_t)q * P + ec]; },
                     acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int k = kt * 16 + 4 * v + h;
            const double lam = lxy + lz[imin(k, nz - 1)];
            fdm_lds[k * kFdm3P + r] = lam > eps ? acc[v] / (s * lam) : 0.0;
        }
    }
    __syncthreads();
    for (int kt = w; kt < gz; kt += NT / 64) {
        const int kc = imin(kt * 16 + r, nz - 1);
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
        mfma_tile<8>(0, nz, [&](int q) { return Wz[q * nz + kc]; }, [&](int q) { return fdm_lds[q * kFdm3P + r]; },
                     acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int k = kt * 16 + 4 * v + h;
            if (k < nz && e < P) data[(int64_t)k * P + e] = acc[v];
        }
    }
}

// The z pass as two launches (INV: the inverse), 64 planes of 16 cells per
// workgroup: for long columns of few cells, which would leave both products of
// a column, and all of the basis, to one CU.
template <bool INV>
__global__ __launch_bounds__(256) void k_fdm3_z_part(int nx, int ny, int nz, const double* in, double* out,
                                                     const double* Vz, const double* lx, const double* ly,
                                                     const double* lz, double s, double eps, const SolverState* st) {
    if (st->done) return;
    const int P = nx * ny, lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, h = lane >> 4;
    const int e = blockIdx.x * 16 + r, ec = imin(e, P - 1), k0 = blockIdx.y * 64 + 16 * w;
    if (k0 >= nz) return;
    const int kc = imin(k0 + r, nz - 1);
    const double* W = INV ? basis_t(Vz, nz) : Vz;
    const double lxy = lx[ec % nx] + ly[ec / nx];
    mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
    mfma_tile<8>(0, nz, [&](int q) { return W[q * nz + kc]; }, [&](int q) { return in[(int64_t)q * P + ec]; }, acc);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int k = k0 + 4 * v + h;
        const double lam = lxy + lz[imin(k, nz - 1)];
        if (k < nz && e < P) out[(int64_t)k * P + e] = INV ? acc[v] : lam > eps ? acc[v] / (s * lam) : 0.0;
    }
}

// inverse y then x of plane K, rows [j0, j0 + 16): in (double) -> out. One tile
// of columns is one wave's chain of loads in y: twice as many in flight then.
template <typename Tout, int NT>
__global__ __launch_bounds__(NT) void k_fdm3_inv(int nx, int ny, const double* in, Tout* out, const double* Vx,
                                                 const double* Vy, const SolverState* st) {
    if (st->done) return;
    extern __shared__ double fdm_lds[];
    const int gy = (ny + 15) >> 4, K = blockIdx.x / gy, j0 = (blockIdx.x - K * gy) * 16, R = fdm3_row(nx);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, h = lane >> 4, gx = (nx + 15) >> 4;
    const int jc = imin(j0 + r, ny - 1);
    const double *Wx = basis_t(Vx, nx), *Wy = basis_t(Vy, ny);
    const double* src = in + (int64_t)K * nx * ny;
    Tout* dst = out + (int64_t)K * nx * ny;
    for (int it = w; it < gx; it += NT / 64) {
        const int ic = imin(it * 16 + r, nx - 1);
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
        auto fa = [&](int q) { return Wy[q * ny + jc]; };
        auto fb = [&](int q) { return src[q * nx + ic]; };
        if (gx == 1 && ny > 64) mfma_tile<16>(0, ny, fa, fb, acc);
        else mfma_tile<8>(0, ny, fa, fb, acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) fdm_lds[(4 * v + h) * R + it * 16 + r] = acc[v];
    }
    __syncthreads();
    for (int it = w; it < gx; it += NT / 64) {
        const int ic = imin(it * 16 + r, nx - 1);
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
        mfma_tile<8>(0, nx, [&](int q) { return fdm_lds[r * R + q]; }, [&](int q) { return Wx[q * nx + ic]; }, acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = j0 + 4 * v + h, i = it * 16 + r;
            if (j < ny && i < nx) dst[j * nx + i] = (Tout)acc[v];
        }
    }
}

// The whole solve of a level of at most 16 cells per axis in one workgroup:
// one plane (x, y) or row of planes (z) per wave, the field and the bases in
// LDS as 16^3 and 16 x 16 entries, zero past the level (no product needs a
// bound). A wave reads its whole plane before it writes it, so the products run
// in place. 8^3 12 us in three launches, 5.6 in this one; 16^3 in f64 8.8.
constexpr int kFdm3One = 16, kFdm3OneThreads = 1024;
template <typename T>
__global__ __launch_bounds__(kFdm3OneThreads) void k_fdm3_one(int nx, int ny, int nz, const T* in, T* out,
                                                              const double* Vx, const double* Vy, const double* Vz,
                                                              const double* lx, const double* ly, const double* lz,
                                                              double s, double eps, const SolverState* st) {
    if (st->done) return;
    constexpr int N = kFdm3One, R = N + 1, PL = N * R;
    __shared__ double a[N * PL], vv[3][PL];
    const int t = threadIdx.x;
    double f[4];
    const int i = t & 15, j = (t >> 4) & 15, k0 = t >> 8;  // cells (k0 + 4 u, j, i)
    const bool in_xy = i < nx && j < ny;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int k = k0 + 4 * u;
        f[u] = in_xy && k < nz ? (double)in[(k * ny + j) * nx + i] : 0.0;
    }
    if (k0 < 3) {
        const int n = k0 == 0 ? nx : k0 == 1 ? ny : nz;
        const double* V = k0 == 0 ? Vx : k0 == 1 ? Vy : Vz;
        vv[k0][j * R + i] = i < n && j < n ? V[j * n + i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) a[(k0 + 4 * u) * PL + j * R + i] = f[u];
    __syncthreads();
    const int w = t >> 6, lane = t & 63, r = lane & 15, h = lane >> 4;
    // out = A B over q of the wave's 16 x 16 entries at o + row * rs + column
    auto product = [&](double* o, int rs, auto fa, auto fb) {
        mfma_d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < N; q += 4) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(fa(q + h), fb(q + h), acc, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[(4 * v + h) * rs + r] = acc[v];
    };
    double* pk = a + w * PL;  // plane k = w
    double* pj = a + w * R;   // row j = w of every plane
    if (w < nz) product(pk, R, [&](int q) { return pk[r * R + q]; }, [&](int q) { return vv[0][q * R + r]; });
    __syncthreads();
    if (w < nz) product(pk, R, [&](int q) { return vv[1][q * R + r]; }, [&](int q) { return pk[q * R + r]; });
    __syncthreads();
    if (w < ny) product(pj, PL, [&](int q) { return vv[2][q * R + r]; }, [&](int q) { return pj[q * PL + r]; });
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int k = k0 + 4 * u;
        double& x = a[k * PL + j * R + i];
        const double lam = in_xy && k < nz ? lx[i] + ly[j] + lz[k] : 0.0;
        x = lam > eps ? x / (s * lam) : 0.0;
    }
    __syncthreads();
    if (w < ny) product(pj, PL, [&](int q) { return vv[2][r * R + q]; }, [&](int q) { return pj[q * PL + r]; });
    __syncthreads();
    if (w < nz) product(pk, R, [&](int q) { return vv[1][r * R + q]; }, [&](int q) { return pk[q * R + r]; });
    __syncthreads();
    if (w < nz) product(pk, R, [&](int q) { return pk[r * R + q]; }, [&](int q) { return vv[0][r * R + q]; });
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int k = k0 + 4 * u;
        if (in_xy && k < nz) out[(k * ny + j) * nx + i] = (T)a[k * PL + j * R + i];
    }
}

// Whether the 3D coarsest level takes the matrix cores (PANO_FDM_SPLIT=0: the
// one-workgroup-per-plane passes, where a plane and a slice fit LDS).
static bool fdm_split_on(const Dims& C) {
    const char* e = getenv("PANO_FDM_SPLIT");
    const bool in_lds = C.w * C.h <= kFdmPlane && C.w * C.d <= kFdmPlane;
    return !in_lds || (C.d > 1 && !(e && e[0] == '0'));
}

// 3D f32 with the fused passes on: the restriction into the coarsest level is
// done by the coarsest solve's first pass (k_fdm_plane_rc) when that level
// takes the in-LDS plane path and the level above restricts a stored residual.
template <typename T, int DIM>
static bool coarse_rc(const MG<T>* m) {
    if constexpr (!std::is_same<T, float>::value || DIM != 3) {
        return false;
    } else {
        if (m->fdm_split) return false;
        const int Lc = m->levels - 1;
        const Dims& C = m->dims[Lc];
        return m->tb && Lc >= 1 && !rr_on(m->tb, m->dims[Lc - 1]) && !leg_on(m, Lc - 1) && C.w * C.h <= kFdmPlane &&
               C.w * C.d <= kFdmPlane;
    }
}

// r: the coarsest right-hand side, or with coarse_rc the fine residual of
// level levels-2 to restrict on the fly.
template <typename T, int DIM>
static pano_status coarse_solve(Ctx* c, MG<T>* m, T* z, const T* r, const SolverState* st) {
    const Dims& C = m->dims[m->levels - 1];
    int nx = C.w, ny = C.h, nz = C.d;
    double s = m->s[m->levels - 1];
    double* t0 = m->fdm_tmp[0];
    double* t1 = m->fdm_tmp[1];
    const double eps = 1e-10;
    hipStream_t S = c->stream;
    const double *Vx = m->fdm_v[0], *Vy = m->fdm_v[1], *Vz = m->fdm_v[2];
    const double *lx = m->fdm_lam[0], *ly = m->fdm_lam[1], *lz = m->fdm_lam[2];
    if (DIM == 2) {
        if (fdm2_one(nx, ny)) {
            hipLaunchKernelGGL((k_fdm2_one<T>), dim3(1), dim3(kFdm2Threads), fdm2_one_lds(nx, ny), S, nx, ny, r, z, Vx,
                               Vy, lx, ly, s, eps, st);
        } else {
            const dim3 G((unsigned)(((nx + 15) / 16) * ((ny + 15) / 16)));
            hipLaunchKernelGGL((k_fdm2_tile<T, double>), G, dim3(256), 0, S, nx, ny, 0, r, t0, Vx, Vy, lx, ly, s, eps,
                               st);
            hipLaunchKernelGGL((k_fdm2_tile<double, double>), G, dim3(256), 0, S, nx, ny, 1, (const double*)t0, t1, Vx,
                               Vy, lx, ly, s, eps, st);
            hipLaunchKernelGGL((k_fdm2_tile<double, double>), G, dim3(256), 0, S, nx, ny, 2, (const double*)t1, t0, Vx,
                               Vy, lx, ly, s, eps, st);
            hipLaunchKernelGGL((k_fdm2_tile<double, T>), G, dim3(256), 0, S, nx, ny, 3, (const double*)t0, z, Vx, Vy,
                               lx, ly, s, eps, st);
        }
        PANO_HIP(hipGetLastError());
        return PANO_OK;
    }
    if (m->fdm_split) {
        if (nx <= kFdm3One && ny <= kFdm3One && nz <= kFdm3One) {
            hipLaunchKernelGGL((k_fdm3_one<T>), dim3(1), dim3(kFdm3OneThreads), 0, S, nx, ny, nz, r, z, Vx, Vy, Vz, lx,
                               ly, lz, s, eps, st);
            PANO_HIP(hipGetLastError());
            return PANO_OK;
        }
        const std::integral_constant<int, 256> nt4{};    // four waves: one tile each up to 64 cells per axis
        const std::integral_constant<int, 1024> nt16{};  // 16 for longer axes
        const unsigned gx = (unsigned)((nx + 15) / 16), gy = (unsigned)((ny + 15) / 16);
        const unsigned gz = (unsigned)((nz + 15) / 16), P16 = (unsigned)((nx * ny + 15) / 16);
        auto fwd = [&](auto nt, unsigned split) {
            hipLaunchKernelGGL((k_fdm3_fwd<T, nt.value>), dim3(nz * gx, split), dim3(nt.value), fdm3_lds_cols(ny), S, nx,
                               ny, r, t0, Vx, Vy, st);
        };
        auto zz = [&](auto nt) {
            hipLaunchKernelGGL(k_fdm3_z<nt.value>, dim3(P16), dim3(nt.value), fdm3_lds_cols(nz), S, nx, ny, nz, t0, Vz,
                               lx, ly, lz, s, eps, st);
        };
        auto inv = [&](auto nt) {
            hipLaunchKernelGGL((k_fdm3_inv<T, nt.value>), dim3(nz * gy), dim3(nt.value),
                               (size_t)16 * fdm3_row(nx) * sizeof(double), S, nx, ny, (const double*)t0, z, Vx, Vy, st);
        };
        if (gy <= 4) fwd(nt4, 1);
        else fwd(nt16, nz * gx < 64 ? (gy + 3) / 4 : 1);
        if (gz <= 4) {
            zz(nt4);
        } else if (P16 > 128) {
            zz(nt16);
        } else {
            const dim3 zg(P16, (gz + 3) / 4);
            hipLaunchKernelGGL(k_fdm3_z_part<false>, zg, dim3(256), 0, S, nx, ny, nz, (const double*)t0, t1, Vz, lx, ly,
                               lz, s, eps, st);
            hipLaunchKernelGGL(k_fdm3_z_part<true>, zg, dim3(256), 0, S, nx, ny, nz, (const double*)t1, t0, Vz, lx, ly,
                               lz, s, eps, st);
        }
        if (gx <= 4) inv(nt4);
        else inv(nt16);
        PANO_HIP(hipGetLastError());
        return PANO_OK;
    }
    const size_t lds = kFdmLdsBytes;
    if constexpr (std::is_same<T, float>::value) {
        if (coarse_rc<T, DIM>(m))
            hipLaunchKernelGGL(k_fdm_plane_rc, dim3(nz), dim3(kFdmThreads), lds, S, m->dims[m->levels - 2], C,
                               (const float*)r, t0, Vx, Vy, s, eps, st);
        else
            hipLaunchKernelGGL((k_fdm_plane<T, double>), dim3(nz), dim3(kFdmThreads), lds, S, nx, ny, 0, r, t0, Vx, Vy,
                               (const double*)nullptr, (const double*)nullptr, s, eps, st);
    } else {
        hipLaunchKernelGGL((k_fdm_plane<T, double>), dim3(nz), dim3(kFdmThreads), lds, S, nx, ny, 0, r, t0, Vx, Vy,
                           (const double*)nullptr, (const double*)nullptr, s, eps, st);
    }
    hipLaunchKernelGGL(k_fdm_zcol, dim3(ny), dim3(kFdmThreads), lds, S, nx, ny, nz, t0, Vz, lx, ly, lz, s, eps, st);
    hipLaunchKernelGGL((k_fdm_plane<double, T>), dim3(nz), dim3(kFdmThreads), lds, S, nx, ny, 1, t0, z, Vx, Vy,
                       (const double*)nullptr, (const double*)nullptr, s, eps, st);
    PANO_HIP(hipGetLastError());
    return PANO_OK;
}

// One level of the V-cycle's down leg: pre-smoothing from z = 0, residual,
// restriction into level l+1. NZ = run_len of the level.
template <typename T, int DIM, int NZ>
static void level_down(Ctx* c, MG<T>* m, int l, T* const* zl, const T* const* rl, const SolverState* st) {
    const int Lc = m->levels - 1;
    const Dims& D = m->dims[l];
    const Dims& Dc = m->dims[l + 1];
    const dim3 B(kTX, kTY);
    const double cfrac = DIM == 3 ? 0.125 : 0.25;
    T s = (T)m->s[l];
    RInv<T> ri = make_rinv<T>(s);
    Grid3 G = grid3_rb(D);
    const double unit = (double)D.d * D.h * D.w * sizeof(T);
    const char* nh = l == 0 ? "smooth_l0" : "";
    if (leg_on(m, l)) {
        // pre-smoothing, residual and restriction in one launch (bytes: r in, the red half of z and r_c out)
        auto down = [&](auto lc) {
            with_leg<DIM>(D, [&](auto th) {
                constexpr int LC = decltype(lc)::value;
                constexpr bool THIN = decltype(th)::value;
                using S = LegS<T, DIM, true, THIN>;
                const LegGrid g = leg_grid<S>(D);
                klaunch(c, l == 0 ? "leg_down_l0" : "", (1.5 + cfrac) * unit, k_leg_down<T, DIM, THIN, LC>, dim3(g.nb),
                        dim3(S::NT), D, Dc, g, zl[l], rl[l], m->r[l + 1], s, ri, st);
            });
        };
        if (l + 1 == Lc) down(std::integral_constant<int, NATURAL>{});
        else down(std::integral_constant<int, REDBLACK>{});
        return;
    }
    // 3D f32, nu = 2: the four half-sweeps from z = 0 in one pass (z is only
    // written, so the pass may write it in place). Timed bytes: the algorithmic
    // bytes of the work, two red-black sweeps of 3 field passes each; the pass
    // itself moves about 2 (b in, z out).
    bool tb_done = false;
    if constexpr (std::is_same<T, float>::value) {
        if (tb_on(m->tb, m->nu, D)) {
            smooth_tb<0, true, false>(c, l == 0 ? "smooth_pre_l0" : "", 6 * unit, D, (const float*)zl[l], zl[l],
                                      rl[l], s, ri, (double*)nullptr, (int*)nullptr, st);
            tb_done = true;
        }
    }
    // first sweep from z = 0: on bandwidth-bound levels red cells then the
    // black half-sweep (two light passes), elsewhere one fused launch
    if (tb_done) {
    } else if (NZ == 4) {
        klaunch(c, l == 0 ? "red_init_l0" : "", unit, k_red_init<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l], rl[l], s,
                ri, st);
        klaunch(c, nh, 1.5 * unit, k_smooth_half<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l], rl[l], s, ri, 1,
                (double*)nullptr, st);
    } else {
        klaunch(c, l == 0 ? "smooth_first_l0" : "", 2 * unit, k_smooth_first<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l],
                rl[l], s, ri, st);
    }
    for (int k = 1; k < m->nu && !tb_done; ++k) {
        klaunch(c, nh, 1.5 * unit, k_smooth_half<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l], rl[l], s, ri, 0,
                (double*)nullptr, st);
        klaunch(c, nh, 1.5 * unit, k_smooth_half<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l], rl[l], s, ri, 1,
                (double*)nullptr, st);
    }
    // f32: residual and restriction in one pass (bytes: z and b in, r_c out) on
    // 3D levels of 2^23 cells and more and on every 2D level
    if constexpr (std::is_same<T, float>::value && DIM == 3) {
        if (rr_on(m->tb, D)) {
            const char* nrr = l == 0 ? "resrestrict_l0" : "";
            if (l + 1 == Lc)
                resrestrict<NATURAL>(c, nrr, (2 + cfrac) * unit, D, Dc, zl[l], rl[l], m->r[l + 1], s, st);
            else
                resrestrict<REDBLACK>(c, nrr, (2 + cfrac) * unit, D, Dc, zl[l], rl[l], m->r[l + 1], s, st);
            return;
        }
    }
    if constexpr (std::is_same<T, float>::value && DIM == 2) {
        if (m->tb) {
            const char* nrr = l == 0 ? "resrestrict_l0" : "";
            if (l + 1 == Lc)
                resrestrict2<NATURAL>(c, nrr, (2 + cfrac) * unit, D, Dc, zl[l], rl[l], m->r[l + 1], s, st);
            else
                resrestrict2<REDBLACK>(c, nrr, (2 + cfrac) * unit, D, Dc, zl[l], rl[l], m->r[l + 1], s, st);
            return;
        }
    }
    klaunch(c, l == 0 ? "residual_l0" : "", 3 * unit, k_mg_residual<T, DIM, NZ>, dim3(G.nb), B, D, G, m->res, zl[l],
            rl[l], s, st);
    if (l + 1 == Lc && coarse_rc<T, DIM>(m)) return;  // restricted by the coarsest solve's first pass
    const char* nr = l == 0 ? "restrict_l0" : "";
    const int nk = restrict_run_len(Dc);
    Grid3 Gc = grid3(Dc.w, Dc.h, (Dc.d + nk - 1) / nk);
    auto restrict_into = [&](auto lc) {
        constexpr int LC = decltype(lc)::value;
        if (nk == 4)
            klaunch(c, nr, (1 + cfrac) * unit, k_restrict<T, DIM, LC, 4>, dim3(Gc.nb), B, D, Dc, Gc, m->r[l + 1],
                    (const T*)m->res, st);
        else if (nk == 2)
            klaunch(c, nr, (1 + cfrac) * unit, k_restrict<T, DIM, LC, 2>, dim3(Gc.nb), B, D, Dc, Gc, m->r[l + 1],
                    (const T*)m->res, st);
        else
            klaunch(c, nr, (1 + cfrac) * unit, k_restrict<T, DIM, LC, 1>, dim3(Gc.nb), B, D, Dc, Gc, m->r[l + 1],
                    (const T*)m->res, st);
    };
    if (l + 1 == Lc) restrict_into(std::integral_constant<int, NATURAL>{});
    else restrict_into(std::integral_constant<int, REDBLACK>{});
}

// One level of the up leg: prolongation from level l+1, post-smoothing; at
// level 0 the last (black, red) pair also yields the partials of z.r. zd: the
// level's z as the down leg left it (zl[l], or m->w[l] when the prolongation
// runs inside the post-smoothing).
template <typename T, int DIM, int NZ>
static void level_up(Ctx* c, MG<T>* m, int l, T* const* zl, const T* zd, const T* const* rl,
                     const SolverState* st, double* dot_part, int* dot_np) {
    const int Lc = m->levels - 1;
    const Dims& D = m->dims[l];
    const Dims& Dc = m->dims[l + 1];
    const dim3 B(kTX, kTY);
    const double cfrac = DIM == 3 ? 0.125 : 0.25;
    T s = (T)m->s[l];
    RInv<T> ri = make_rinv<T>(s);
    Grid3 G = grid3_rb(D);
    const double unit = (double)D.d * D.h * D.w * sizeof(T);
    const char* nh = l == 0 ? "smooth_l0" : "";
    const char* np = l == 0 ? "prolong_l0" : "";
    if (leg_up_on(m, l)) {
        // prolongation and post-smoothing in one launch (bytes: the red half of z, z_c and r in, z out)
        const bool dot = l == 0 && dot_part;
        auto up = [&](auto lc, auto dt) {
            with_leg<DIM>(D, [&](auto th) {
                constexpr int LC = decltype(lc)::value;
                constexpr bool DOT = decltype(dt)::value, THIN = decltype(th)::value;
                using S = LegS<T, DIM, false, THIN>;
                const LegGrid g = leg_grid<S>(D);
                klaunch(c, l == 0 ? "leg_up_l0" : "", (2.5 + cfrac) * unit, k_leg_up<T, DIM, THIN, LC, DOT>,
                        dim3(g.nb), dim3(S::NT), D, Dc, g, zd, zl[l], rl[l], (const T*)zl[l + 1], s, ri, dot_part, st);
                if (DOT) *dot_np = 2 * g.nb;
            });
        };
        auto up_lc = [&](auto lc) {
            if (dot) up(lc, std::true_type{});
            else up(lc, std::false_type{});
        };
        if (l + 1 == Lc) up_lc(std::integral_constant<int, NATURAL>{});
        else up_lc(std::integral_constant<int, REDBLACK>{});
        return;
    }
    // f32 with the prolongation in the post-smoothing: the four half-sweeps
    // from zd + P z_{l+1} into z in one pass (zd: the pre-smoothed z, a
    // separate buffer, as other workgroups still read their halo from it while
    // this one stores). Timed bytes: the prolongation pass (z and z_c in, z
    // out) and two red-black sweeps of 3 field passes each; the pass moves
    // about 3.
    if constexpr (std::is_same<T, float>::value) {
        if (zd != zl[l]) {
            const char* npost = l == 0 ? "smooth_post_l0" : "";
            const double bytes = (8 + cfrac) * unit;
            const bool dot = l == 0 && dot_part;
            auto post = [&](auto lc) {
                constexpr int LC = decltype(lc)::value;
                if (dot)
                    smooth_tb<1, false, true, LC>(c, npost, bytes, D, (const float*)zd, zl[l], rl[l], s, ri,
                                                  dot_part, dot_np, st, (const float*)zl[l + 1], Dc);
                else
                    smooth_tb<1, false, false, LC>(c, npost, bytes, D, (const float*)zd, zl[l], rl[l], s, ri,
                                                   (double*)nullptr, (int*)nullptr, st, (const float*)zl[l + 1],
                                                   Dc);
            };
            if (l + 1 == Lc) post(std::integral_constant<int, NATURAL>{});
            else post(std::integral_constant<int, REDBLACK>{});
            return;
        }
    }
    // f32, nu = 2: prolongation into the residual scratch (free on the up
    // leg), then the four post-smoothing half-sweeps from there back into z in
    // one pass (out of place: workgroups read their halo from the input while
    // others store). Timed bytes: two red-black sweeps of 3 field passes each;
    // the pass moves about 3.
    bool tb = false;
    if constexpr (std::is_same<T, float>::value) tb = tb_on(m->tb, m->nu, D);
    T* zo = tb ? m->res : zl[l];
    if constexpr (DIM == 3 && std::is_same<T, float>::value) {
        if (l + 1 == Lc)
            klaunch(c, np, (2 + cfrac) * unit, k_prolong3_lds<NATURAL, NZ>, dim3(G.nb), B, D, Dc, G, zo,
                    (const T*)zl[l], (const T*)m->z[l + 1], st);
        else
            klaunch(c, np, (2 + cfrac) * unit, k_prolong3_lds<REDBLACK, NZ>, dim3(G.nb), B, D, Dc, G, zo,
                    (const T*)zl[l], (const T*)m->z[l + 1], st);
    } else if (l + 1 == Lc) {
        klaunch(c, np, (2 + cfrac) * unit, k_prolong<T, DIM, NATURAL, NZ>, dim3(G.nb), B, D, Dc, G, zo,
                (const T*)zl[l], (const T*)m->z[l + 1], st);
    } else {
        klaunch(c, np, (2 + cfrac) * unit, k_prolong<T, DIM, REDBLACK, NZ>, dim3(G.nb), B, D, Dc, G, zo,
                (const T*)zl[l], (const T*)m->z[l + 1], st);
    }
    if constexpr (std::is_same<T, float>::value) {
        if (tb) {
            const char* npost = l == 0 ? "smooth_post_l0" : "";
            if (l == 0 && dot_part)
                smooth_tb<1, false, true>(c, npost, 6 * unit, D, (const float*)zo, zl[l], rl[l], s, ri, dot_part,
                                          dot_np, st);
            else
                smooth_tb<1, false, false>(c, npost, 6 * unit, D, (const float*)zo, zl[l], rl[l], s, ri,
                                           (double*)nullptr, (int*)nullptr, st);
            return;
        }
    }
    for (int k = 0; k < m->nu; ++k) {
        bool last = l == 0 && k == m->nu - 1 && dot_part;
        double* pb = last ? dot_part : nullptr;
        double* pr = last ? dot_part + G.nb : nullptr;
        klaunch(c, nh, 1.5 * unit, k_smooth_half<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l], rl[l], s, ri, 1, pb, st);
        klaunch(c, nh, 1.5 * unit, k_smooth_half<T, DIM, NZ>, dim3(G.nb), B, D, G, zl[l], rl[l], s, ri, 0, pr, st);
        if (last) *dot_np = 2 * G.nb;
    }
}

template <typename T, int DIM>
static pano_status vcycle_dim(Ctx* c, MG<T>* m, T* z0, const T* r0, const SolverState* st, double* dot_part,
                              int* dot_np) {
    int Lc = m->levels - 1;
    T* zl[16];
    const T* rl[16];
    zl[0] = z0;
    rl[0] = r0;
    for (int l = 1; l <= Lc; ++l) {
        zl[l] = m->z[l];
        rl[l] = m->r[l];
    }
    // the down leg's z: the pre-smoothing's output, read by the residual and
    // (with the prolongation in the post-smoothing) by the post-smoothing
    T* zd[16];
    for (int l = 0; l <= Lc; ++l) zd[l] = l < Lc && m->w[l] ? m->w[l] : zl[l];
    for (int l = 0; l < Lc; ++l) {
        switch (run_len(m->dims[l])) {
            case 4: level_down<T, DIM, 4>(c, m, l, zd, rl, st); break;
            case 2: level_down<T, DIM, 2>(c, m, l, zd, rl, st); break;
            default: level_down<T, DIM, 1>(c, m, l, zd, rl, st); break;
        }
    }
    PANO_CHECK(coarse_solve<T, DIM>(c, m, m->z[Lc], coarse_rc<T, DIM>(m) ? (const T*)m->res : m->r[Lc], st));
    for (int l = Lc - 1; l >= 0; --l) {
        switch (run_len(m->dims[l])) {
            case 4: level_up<T, DIM, 4>(c, m, l, zl, zd[l], rl, st, dot_part, dot_np); break;
            case 2: level_up<T, DIM, 2>(c, m, l, zl, zd[l], rl, st, dot_part, dot_np); break;
            default: level_up<T, DIM, 1>(c, m, l, zl, zd[l], rl, st, dot_part, dot_np); break;
        }
    }
    PANO_HIP(hipGetLastError());
    return PANO_OK;
}

int mg_leg_blocks(const Dims& D) {
    if (D.d <= 1) return leg_grid<LegS<double, 2, false, false>>(D).nb;
    return leg_thin(D) ? leg_grid<LegS<double, 3, false, true>>(D).nb : leg_grid<LegS<double, 3, false, false>>(D).nb;
}

template <typename T>
pano_status mg_vcycle(Ctx* c, MG<T>* m, T* z0, const T* r0, const SolverState* st, double* dot_part,
                      int* dot_np) {
    if (m->dims[0].d > 1) return vcycle_dim<T, 3>(c, m, z0, r0, st, dot_part, dot_np);
    return vcycle_dim<T, 2>(c, m, z0, r0, st, dot_part, dot_np);
}

template pano_status mg_setup<float>(Ctx*, const Dims&, int, int, double, MG<float>*);
template pano_status mg_setup<double>(Ctx*, const Dims&, int, int, double, MG<double>*);
template pano_status mg_vcycle<float>(Ctx*, MG<float>*, float*, const float*, const SolverState*, double*, int*);
template pano_status mg_vcycle<double>(Ctx*, MG<double>*, double*, const double*, const SolverState*, double*,
                                        int*);

}  // namespace pano
