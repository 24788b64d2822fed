// The two legs of a V-cycle level as one launch each, for levels whose time is
// launches and latency rather than bytes:
//  down: the four pre-smoothing half-sweeps from z = 0, the residual and its
//        restriction (three launches before: 15.5 us at 64^3, 9.8 us now);
//  up:   the prolongation added to the pre-smoothed z, the four post-smoothing
//        half-sweeps and the sums of z.r (13.6 us at 64^3 in one streaming
//        launch, 9.2 us now).
//
// A workgroup owns a tile of TXP x-pairs by TY rows by TZ planes and holds the
// tile and its halo at once (no plane-by-plane stream: its steps are a chain
// of barriers that small levels have too few workgroups to hide). A thread
// owns one column of pairs over a group of planes: both colours of its z and b
// in registers, so of the six neighbours of a cell three come from its own
// registers (the other cell of the pair and the two planes) and three from
// LDS (the next pair and the two rows), where colour c of plane l, column t is
// word (c * PZ + l) * CT + t: consecutive lanes, consecutive words.
//
// Half-sweep h covers the tile grown by as many cells as the later half-sweeps
// and, in the down leg, the restriction's support reach; halo cells are
// recomputed by each neighbouring workgroup with the same arithmetic. Cells
// outside the grid hold 0, what a missing neighbour adds to the sum.
//
// A half-sweep does not read the cell it updates, so the up leg needs only the
// red cells of z + P z_c: the black ones are overwritten first. The down leg
// therefore stores the red half of z alone.
//
// Values are the expressions of the half-sweep, residual, restriction and
// prolongation kernels on the same operands in the same order, so a level's
// result has their bits (z.r sums are added in another order).
#pragma once

#include "mg_device.hpp"

namespace pano {

template <typename T, int DIM, int TXP_, int TY_, int TZ_, bool DOWN>
struct LegShape {
    static constexpr int TXP = TXP_, TY = TY_, TZ = TZ_;
    static_assert(TY % 2 == 0 && (DIM == 3 ? TZ % 2 == 0 : TZ == 1), "even tiles");
    static constexpr int H = DOWN ? 5 : 4;             // halo cells
    static constexpr int HP = (H + 1) / 2;             // halo pairs in x
    static constexpr int HZ = DIM == 3 ? H : 0;
    static constexpr int PX = TXP + 2 * HP, PY = TY + 2 * H, PZ = TZ + 2 * HZ;
    static constexpr int COLS = PX * PY, CT = (COLS + 63) / 64 * 64;  // columns, in whole waves
    // thread groups along z, an even number of planes each (with one group a
    // SIMD's one wave waits for LDS and its own results at every instruction:
    // 64^3 down leg 12.5 us with one group of 18 planes, 9.8 with three of 6)
    static constexpr int G = DIM == 2 ? 1 : DOWN ? PZ / (PZ % 6 == 0 && PZ > 12 ? 6 : 4) : PZ / (PZ % 4 == 0 ? 4 : 2), PG = PZ / G, NT = CT * G;
    static_assert(PG * G == PZ && (DIM == 2 || PG % 2 == 0), "whole groups");
    static_assert(NT <= 1024, "one thread per column and group");
    static constexpr int D0 = DOWN ? 5 : 3;            // distance that half-sweep 0 covers; h: D0 - h
    static constexpr int EDGE = PX + 1;                // readable words before and after the columns
    static constexpr int ZW = 2 * PZ * CT + 2 * EDGE;  // LDS: z, or (down) the residual
    // down: the x-y restricted planes
    static constexpr int CX = TXP, CY = TY / 2, CZ = DIM == 3 ? TZ / 2 : 1, NP = DIM == 3 ? 2 * CZ + 2 : 1;
    // up: the coarse region under the tile and halo, one cell more on each side
    static constexpr int RX = PX + 2, RY = PY / 2 + 2, RZ = DIM == 3 ? PZ / 2 + 2 : 1;
    static constexpr int XW = DOWN ? (DIM == 3 ? NP * CX * CY : 0) : RX * RY * RZ;
    static constexpr size_t LDS = (size_t)(ZW + XW) * sizeof(T);
};

struct LegGrid {
    int gx, gy, gz, nb;
};
template <class S>
inline LegGrid leg_grid(const Dims& D) {
    LegGrid g;
    g.gx = ((D.w >> 1) + S::TXP - 1) / S::TXP;
    g.gy = (D.h + S::TY - 1) / S::TY;
    g.gz = (D.d + S::TZ - 1) / S::TZ;
    g.nb = g.gx * g.gy * g.gz;
    return g;
}

// What both legs share: the thread's column and the half-sweeps.
template <typename T, int DIM, class S>
struct LegThread {
    static constexpr int PZ = S::PZ, CT = S::CT, PG = S::PG, PX = S::PX, HZ = S::HZ;
    Dims D;
    T* zl;       // LDS, word 0 of the columns
    T s;
    int t, l0;                 // the column, the group's first plane (uniform across a wave)
    int mp, row, m, y, z0;     // z0: the tile's first plane
    int yp;      // y & 1
    bool ind;    // the column lies in the grid
    int dx;      // the LDS step to the x neighbour outside the pair, of a cell of x parity yp; -dx for the other
    int dist[2]; // how far the cell of x parity (k ^ yp) lies outside the tile, in x and y
    int nxy[2];  // its x and y neighbours that are not walls
    unsigned off, hw, n2;  // in-plane offset (0 outside the grid), plane and colour strides
    T v[2][PG], b[2][PG];      // of planes l0 + q

    __device__ __forceinline__ void init(T* lds, const Dims& D_, int bx, int by, int bz, T s_) {
        D = D_;
        s = s_;
        t = threadIdx.x % CT;
        l0 = DIM == 2 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / CT) * PG;
        zl = lds + S::EDGE;
        const int tt = t < S::COLS ? t : 0;
        mp = tt % PX;
        row = tt / PX;
        m = bx * S::TXP - S::HP + mp;
        y = by * S::TY - S::H + row;
        z0 = bz * S::TZ;
        yp = y & 1;
        const int wh = D.w >> 1;
        ind = t < S::COLS && m >= 0 && m < wh && y >= 0 && y < D.h;
        dx = yp ? 1 : -1;
        off = ind ? (unsigned)(y * wh + m) : 0u;
        hw = (unsigned)(D.h * wh);
        n2 = (unsigned)D.d * hw;
        const int dy = row < S::H ? S::H - row : row >= S::H + S::TY ? row - (S::H + S::TY - 1) : 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int p = k ^ yp, xl = 2 * mp + p, x = 2 * m + p;
            const int dd = xl < 2 * S::HP ? 2 * S::HP - xl : xl >= 2 * (S::HP + S::TXP) ? xl - 2 * (S::HP + S::TXP) + 1 : 0;
            dist[k] = ind ? (dd > dy ? dd : dy) : 64;
            const int hxy = (x > 0) | ((x < D.w - 1) << 1) | ((y > 0) << 2) | ((y < D.h - 1) << 3);
            nxy[k] = __builtin_popcount((unsigned)((hxy | D.bc) & 0xF));
        }
    }
    // plane l of the column arrays: its z (clamped for loads), whether it is in the grid
    __device__ __forceinline__ int z_of(int l) const { return z0 - HZ + l; }
    __device__ __forceinline__ bool in_z(int l) const { return DIM == 2 || (z_of(l) >= 0 && z_of(l) < D.d); }
    __device__ __forceinline__ const T* plane(const T* f, int c, int l) const {
        const int z = DIM == 2 ? 0 : imin(imax(z_of(l), 0), D.d - 1);
        return f + (size_t)(c ? n2 : 0u) + (size_t)z * hw;
    }
    // distance of plane l from the tile's planes
    static __device__ __forceinline__ int dz(int l) { return DIM == 2 ? 0 : l < HZ ? HZ - l : l >= HZ + S::TZ ? l - (HZ + S::TZ - 1) : 0; }
    // parity of the z of plane l0 + q (z0, l0 even)
    static constexpr int zpar(int q) { return DIM == 2 ? 0 : (q + HZ) & 1; }
    __device__ __forceinline__ T* word(int c, int l) const { return zl + (c * PZ + l) * CT + t; }

    // z neighbours of plane l that are not walls
    __device__ __forceinline__ int nz_of(int l) const {
        if (DIM == 2) return 0;
        const int z = z_of(l);
        return (z > 0 || (D.bc & 16)) + (z < D.d - 1 || (D.bc & 32));
    }
    // sum of the neighbours (colour 1 - c) of the column's colour-c cell on
    // plane l0 + q (not the region's first or last plane)
    template <int C>
    __device__ __forceinline__ T nbr_sum(int q) const {
        constexpr int O = 1 - C;
        const T* w = word(O, l0 + q);
        const int step = ((C + zpar(q)) & 1) ? -dx : dx;
        T sum = ((w[step] + v[O][q]) + w[-PX]) + w[PX];
        if constexpr (DIM == 3) {  // a plane of the next group: from LDS
            sum = sum + (q > 0 ? v[O][q > 0 ? q - 1 : 0] : w[-CT]);
            sum = sum + (q < PG - 1 ? v[O][q < PG - 1 ? q + 1 : 0] : w[CT]);
        }
        return sum;
    }
    // half-sweep h (colour C) and the LDS copy of its colour. FIRST: z = 0.
    template <int C, int HS, bool FIRST, bool DOT>
    __device__ __forceinline__ void sweep(const RInv<T>& ri, double& acc) {
        constexpr int DS = S::D0 - HS;
        // reciprocals for x parity class k and two or one z neighbours
        T a[2][2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            a[k][0] = pick(ri, nxy[k] + (DIM == 3 ? 2 : 0));
            a[k][1] = DIM == 3 ? pick(ri, nxy[k] + 1) : a[k][0];
        }
#pragma unroll
        for (int q = 0; q < PG; ++q) {
            const int l = l0 + q;
            if (dz(l) > DS || !in_z(l)) continue;
            const int k = (C + zpar(q)) & 1;
            const T ar = DIM == 3 && nz_of(l) < 2 ? a[k][1] : a[k][0];
            const T sum = FIRST ? (T)0 : nbr_sum<C>(q);
            const T nv = (b[C][q] + s * sum) * ar;
            const bool on = dist[k] <= DS;
            v[C][q] = on ? nv : v[C][q];
            if (DOT && dz(l) == 0) acc += dist[k] == 0 ? (double)nv * (double)b[C][q] : 0.0;
            *word(C, l) = v[C][q];
        }
    }
    static __device__ __forceinline__ T pick(const RInv<T>& ri, int nc) {
        T r = ri.v[1];
#pragma unroll
        for (int q = 2; q <= 6; ++q) r = nc == q ? ri.v[q] : r;
        return r;
    }
};

// Down leg of tile (bx, by, bz): z (red half) into zo, r_c into rc.
template <typename T, int DIM, class S, int LC>
__device__ __forceinline__ void leg_down(T* lds, const Dims& D, const Dims& Dc, int bx, int by, int bz, T* zo,
                                         const T* r, T* rc, T s, const RInv<T>& ri) {
    LegThread<T, DIM, S> th;
    th.init(lds, D, bx, by, bz, s);
    constexpr int PZ = S::PZ, PG = S::PG, HZ = S::HZ, PX = S::PX, CT = S::CT, NT = S::NT;
#pragma unroll
    for (int q = 0; q < PG; ++q) {
        th.b[0][q] = th.plane(r, 0, th.l0 + q)[th.off];
        th.b[1][q] = th.plane(r, 1, th.l0 + q)[th.off];
        th.v[0][q] = th.v[1][q] = (T)0;
    }
#pragma unroll
    for (int q = 0; q < PG; ++q) *th.word(0, th.l0 + q) = *th.word(1, th.l0 + q) = (T)0;
    double none = 0.0;
    th.template sweep<0, 0, true, false>(ri, none);
    __syncthreads();
    th.template sweep<1, 1, false, false>(ri, none);
    __syncthreads();
    th.template sweep<0, 2, false, false>(ri, none);
    __syncthreads();
    th.template sweep<1, 3, false, false>(ri, none);
    __syncthreads();
    // the tile's red cells, and the residual over the tile and one cell around
    // it, which then takes the place of z in LDS
    const bool own = th.ind && th.mp >= S::HP && th.mp < S::HP + S::TXP && th.row >= S::H && th.row < S::H + S::TY;
    constexpr int L0 = DIM == 3 ? HZ - 1 : 0;  // first plane of the restriction's support
    T res[2][PG];
#pragma unroll
    for (int q = 0; q < PG; ++q) {
        const int l = th.l0 + q;
        res[0][q] = res[1][q] = (T)0;
        if (th.dz(l) > 1) continue;
        if (own && th.dz(l) == 0 && th.in_z(l)) zo[(size_t)th.z_of(l) * th.hw + th.off] = th.v[0][q];
        const int nz = th.nz_of(l);
        const T n0 = (T)(th.nxy[(0 + th.zpar(q)) & 1] + nz), n1 = (T)(th.nxy[(1 + th.zpar(q)) & 1] + nz);
        const T a0 = s * (n0 * th.v[0][q] - th.template nbr_sum<0>(q));
        const T a1 = s * (n1 * th.v[1][q] - th.template nbr_sum<1>(q));
        res[0][q] = th.b[0][q] - a0;
        res[1][q] = th.b[1][q] - a1;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PG; ++q) {
        if (th.dz(th.l0 + q) > 1) continue;
        *th.word(0, th.l0 + q) = res[0][q];
        *th.word(1, th.l0 + q) = res[1][q];
    }
    __syncthreads();
    // x, then y restriction of fine plane l over coarse column (i, j) of the tile
    const int I0 = bx * S::TXP, J0 = by * S::CY, K0 = bz * S::CZ;
    auto restrict_xy = [&](int l, int i, int j) {
        const int I = I0 + i, J = J0 + j;
        const bool hmI = I > 0, hpI = I < Dc.w - 1, hmJ = J > 0, hpJ = J < Dc.h - 1;
        T u[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int rw = S::H + 2 * j - 1 + q;                                // region row of fine y = 2J - 1 + q
            const int ce = (2 * J - 1 + q + (DIM == 3 ? th.z_of(l) : 0)) & 1;  // colour of the even fine x
            const T* pe = th.zl + (ce * PZ + l) * CT + rw * PX + S::HP + i;
            const T* po = th.zl + ((1 - ce) * PZ + l) * CT + rw * PX + S::HP + i;
            u[q] = r1(po[-1], pe[0], po[0], pe[1], hmI, hpI);
        }
        return r1(u[0], u[1], u[2], u[3], hmJ, hpJ);
    };
    constexpr int CXY = S::CX * S::CY;
    if constexpr (DIM == 2) {
        for (int o = threadIdx.x; o < CXY; o += NT) {
            const int i = o % S::CX, j = o / S::CX;
            if (I0 + i < Dc.w && J0 + j < Dc.h) rc[cidx<LC>(Dc, 0, J0 + j, I0 + i)] = restrict_xy(0, i, j);
        }
    } else {
        T* ty = lds + S::ZW;
        for (int o = threadIdx.x; o < S::NP * CXY; o += NT) {
            const int p = o / CXY, e = o - p * CXY;
            ty[o] = restrict_xy(L0 + p, e % S::CX, e / S::CX);
        }
        __syncthreads();
        for (int o = threadIdx.x; o < S::CZ * CXY; o += NT) {
            const int k = o / CXY, e = o - k * CXY, i = e % S::CX, j = e / S::CX, K = K0 + k;
            if (I0 + i < Dc.w && J0 + j < Dc.h && K < Dc.d) {
                const T* q = ty + 2 * k * CXY + e;
                rc[cidx<LC>(Dc, K, J0 + j, I0 + i)] =
                    r1(q[0], q[CXY], q[2 * CXY], q[3 * CXY], K > 0, K < Dc.d - 1);
            }
        }
    }
}

// Up leg of tile (bx, by, bz): zo from zd (red half) + P zc; with DOT acc gets
// the tile's sums of z.r of the last two half-sweeps.
template <typename T, int DIM, class S, int LC, bool DOT>
__device__ __forceinline__ void leg_up(T* lds, const Dims& D, const Dims& Dc, int bx, int by, int bz, const T* zd,
                                       T* zo, const T* r, const T* zc, T s, const RInv<T>& ri, double* acc) {
    LegThread<T, DIM, S> th;
    th.init(lds, D, bx, by, bz, s);
    constexpr int PG = S::PG, HZ = S::HZ, NT = S::NT, RX = S::RX, RY = S::RY;
    const int Ib = bx * S::TXP - S::HP - 1, Jb = by * (S::TY / 2) - S::H / 2 - 1,
              Kb = DIM == 3 ? (th.z0 - HZ) / 2 - 1 : 0;  // z0 - HZ is even
    T* cr = lds + S::ZW;
    {   // every load first: the coarse region (clamped), the red z and b
        constexpr int NC = (S::XW + NT - 1) / NT;
        T cv[NC];
#pragma unroll
        for (int q = 0; q < NC; ++q) {
            const int e = imin((int)threadIdx.x + q * NT, S::XW - 1);
            const int i = e % RX, j = e / RX % RY, k = e / (RX * RY);
            cv[q] = zc[cidx<LC>(Dc, DIM == 3 ? imin(imax(Kb + k, 0), Dc.d - 1) : 0, imin(imax(Jb + j, 0), Dc.h - 1),
                                imin(imax(Ib + i, 0), Dc.w - 1))];
        }
#pragma unroll
        for (int q = 0; q < PG; ++q) {
            th.v[0][q] = th.plane(zd, 0, th.l0 + q)[th.off];
            th.v[1][q] = (T)0;
            th.b[0][q] = th.plane(r, 0, th.l0 + q)[th.off];
            th.b[1][q] = th.plane(r, 1, th.l0 + q)[th.off];
        }
#pragma unroll
        for (int q = 0; q < NC; ++q)
            if ((int)threadIdx.x + q * NT < S::XW) cr[threadIdx.x + q * NT] = cv[q];
    }
    __syncthreads();
    {   // red z + P z_c: Q of a coarse plane for both cells of the pair, then the z weights
        const T w34 = (T)0.75, w14 = (T)0.25, one = (T)1, zero = (T)0;
        const int J = th.yp ? (th.y >> 1) + 1 : (th.y >> 1) - 1;  // the second coarse row of p1
        const bool ey = J < 0 || J >= Dc.h, el = th.m == 0, er = th.m + 1 >= Dc.w;
        const T wy0 = ey ? one : w34, wy1 = ey ? zero : w14;
        const T wl0 = el ? one : w34, wl1 = el ? zero : w14;
        const T wr0 = er ? one : w34, wr1 = er ? zero : w14;
        constexpr int NQ = DIM == 3 ? PG / 2 + 2 : 1;  // coarse planes under the group's planes
        const T* c0 = cr + (th.l0 / 2) * (RX * RY) + ((th.row >> 1) + 1) * RX + th.mp + 1;
        const int dj = th.yp ? RX : -RX;
        T Q[NQ][2];
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            const T* p0 = c0 + k * RX * RY;
            const T* p1_ = p0 + dj;
            const T l0 = wl0 * p0[0] + wl1 * p0[-1], r0 = wr0 * p0[0] + wr1 * p0[1];
            const T l1 = wl0 * p1_[0] + wl1 * p1_[-1], r1_ = wr0 * p1_[0] + wr1 * p1_[1];
            Q[k][0] = wy0 * l0 + wy1 * l1;
            Q[k][1] = wy0 * r0 + wy1 * r1_;
        }
#pragma unroll
        for (int q = 0; q < PG; ++q) {
            const int l = th.l0 + q, sp = th.zpar(q);  // x parity of the red cell: sp ^ yp
            T add;
            if constexpr (DIM == 3) {
                // z = 2 (Kb + 1) + l, l0 even: K0 = Q plane q / 2 + 1, K1 the next one of the other side
                constexpr int M = NQ - 1;
                const int k0 = q / 2 + 1 < M ? q / 2 + 1 : M, k1 = (q & 1) ? (k0 < M ? k0 + 1 : M) : k0 - 1;
                const int z = th.z_of(l), K = (z & 1) ? (z >> 1) + 1 : (z >> 1) - 1;
                const bool ez = K < 0 || K >= Dc.d;
                const T wz0 = ez ? one : w34, wz1 = ez ? zero : w14;
                const T q0 = (sp ^ th.yp) ? Q[k0][1] : Q[k0][0], q1 = (sp ^ th.yp) ? Q[k1][1] : Q[k1][0];
                add = wz0 * q0 + wz1 * q1;
            } else {
                add = th.yp ? Q[0][1] : Q[0][0];
            }
            const T val = th.v[0][q] + add;
            th.v[0][q] = th.ind && th.in_z(l) ? val : (T)0;
            *th.word(0, l) = th.v[0][q];
            *th.word(1, l) = (T)0;
        }
    }
    double none = 0.0;
    __syncthreads();
    th.template sweep<1, 0, false, false>(ri, none);
    __syncthreads();
    th.template sweep<0, 1, false, false>(ri, none);
    __syncthreads();
    th.template sweep<1, 2, false, DOT>(ri, acc[0]);
    __syncthreads();
    th.template sweep<0, 3, false, DOT>(ri, acc[1]);
    const bool own = th.ind && th.mp >= S::HP && th.mp < S::HP + S::TXP && th.row >= S::H && th.row < S::H + S::TY;
#pragma unroll
    for (int q = 0; q < PG; ++q) {
        const int l = th.l0 + q;
        if (own && th.dz(l) == 0 && th.in_z(l)) {
            T* o = zo + (size_t)th.z_of(l) * th.hw + th.off;
            o[0] = th.v[0][q];
            o[th.n2] = th.v[1][q];
        }
    }
}

}  // namespace pano
