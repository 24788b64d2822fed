// CG loop of small natural-layout solves in one kernel (panopaea/src/pcg.rs:48-79).
//
// A 128^2 Jacobi iteration takes seven launches of 3 to 4 us each and almost
// no work in any of them (24.6 us per iteration; 4.6 here). A cluster of up to
// 256 workgroups runs the loop: workgroup g owns the consecutive cells
// [g*chunk, (g+1)*chunk) of the field (whole rows or not), with x and r of its
// cells in registers and p in LDS together with the row before and the row
// after (in 3D the p of the planes above and below in registers of the thread
// whose cell they touch). The halo's p is not exchanged: every workgroup
// computes it from the neighbours' r with the owner's expression, so one
// iteration has two exchanges only, p.q and (z.r, max|r|, edges of r).
//
// An exchange is one hop and every value is its own flag: a workgroup stores
// its FP64 sum into its own slot (and the edges of r into hb) with agent-scope
// stores, which pass the XCDs' L2s, so no cache is written back or
// invalidated; readers poll until no value is the empty mark, a NaN pattern
// that no result has (a NaN is stored as the canonical one). Each thread polls
// at most one slot and the edge values that it needs itself. The slots have
// kClCopies mailboxes, one for the workgroups of each XCD (dispatched in
// turn), all written by every workgroup: readers of one address wait for each
// other (128^2: 5.8 us per iteration with one mailbox, 4.7 with 8, 4.6 with 32).
// Copies: two of hb, z.r and max|r|, four of p.q. Once the p.q exchange of
// iteration k is over for a whole workgroup (behind the barrier after the
// poll: each wave polls 64 slots only), everybody has left iteration k - 1, so
// its copies are emptied there; those stores have completed (s_waitcnt) before
// the workgroup's next p.q is stored, which everybody waits for before a copy
// emptied here is polled again.
//
// Sums are FP64 as in the launches' partials, in another order. Everything
// else is the launches' arithmetic, cell by cell.
//
// Workgroups must run together. The clusters of one process together have at
// most one workgroup per CU (ClReserve), and every wait is bounded all the
// same (another process may hold the CUs): a workgroup that
// polls `spin` times without an answer sets the stop word and the state's
// stalled flag and ends, as does everybody who sees the word; the host then
// takes the launches from the beginning.
#include "cg_cluster.hpp"

#include <condition_variable>
#include <mutex>

namespace pano {

constexpr unsigned long long kClEmpty = 0x7FF8C0DEC0DEC0DEull;
constexpr unsigned long long kClNan = 0x7FF8000000000000ull;

template <typename V>
__device__ __forceinline__ V ld_agent(const V* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename V>
__device__ __forceinline__ void st_agent(V* p, V v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// every store this wave has issued is complete
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// lane exchange within rows of 16 lanes (DPP: no LDS round trip)
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double lane_of(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// quads by lane^1 and lane^2, then the mirrored half row and row, then the four rows
struct ClSum {
    static __device__ __forceinline__ double op(double a, double b) { return a + b; }
};
struct ClMax {
    static __device__ __forceinline__ double op(double a, double b) { return nan_max(a, b); }
};
template <typename OP>
__device__ __forceinline__ double wave_all(double v) {
    v = OP::op(v, dpp<0xB1>(v));
    v = OP::op(v, dpp<0x4E>(v));
    v = OP::op(v, dpp<0x141>(v));
    v = OP::op(v, dpp<0x140>(v));
    return OP::op(OP::op(lane_of(v, 0), lane_of(v, 16)), OP::op(lane_of(v, 32), lane_of(v, 48)));
}

template <typename OP, int NW>
__device__ __forceinline__ double waves_all(const double* r) {
    double v = r[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) v = OP::op(v, r[i]);
    return v;
}

__device__ __forceinline__ unsigned long long cl_bits(double v) {
    return v == v ? (unsigned long long)__double_as_longlong(v) : kClNan;
}

// Thread t < P polls slot t of one or two arrays until its wave has all of
// them; false after `spin` polls or once the stop word is set.
template <int N>
__device__ __forceinline__ bool cl_poll(const unsigned long long* s0, const unsigned long long* s1,
                                        const unsigned long long* stop, int P, unsigned spin, double* v) {
    const int i = threadIdx.x < P ? threadIdx.x : P - 1;
    v[0] = 0.0;
    if (N > 1) v[1] = 0.0;
    if ((int)(threadIdx.x & ~63u) >= P) return true;  // no slot for this wave
    for (unsigned k = 0; k < spin; ++k) {
        const unsigned long long a = ld_agent(s0 + i), b = N > 1 ? ld_agent(s1 + i) : a;
        if (!__any(a == kClEmpty || b == kClEmpty)) {
            v[0] = threadIdx.x < P ? __longlong_as_double((long long)a) : 0.0;
            if (N > 1) v[1] = threadIdx.x < P ? __longlong_as_double((long long)b) : 0.0;
            return true;
        }
        if ((k & 63) == 63 && ld_agent(stop) != 0) return false;
    }
    return false;
}

// The edge values as words: the empty mark and the canonical NaN of T.
template <typename T>
struct ClWord;
template <>
struct ClWord<float> {
    using U = unsigned;
    static constexpr U empty = 0x7FC0DEDEu, nan = 0x7FC00000u;
};
template <>
struct ClWord<double> {
    using U = unsigned long long;
    static constexpr U empty = kClEmpty, nan = kClNan;
};
template <typename T>
__device__ __forceinline__ void edge_store(T* p, T v) {
    typename ClWord<T>::U u = ClWord<T>::nan;
    if (v == v) __builtin_memcpy(&u, &v, sizeof(T));
    st_agent((typename ClWord<T>::U*)p, u);
}
template <typename T>
__device__ __forceinline__ void edge_empty(T* p) {
    st_agent((typename ClWord<T>::U*)p, (typename ClWord<T>::U)ClWord<T>::empty);
}
// Loads N edge values (on: wanted) until all are there, all loads of a try in
// flight together; false when given up.
template <typename T, int N>
__device__ __forceinline__ bool edge_poll(const T* hb, const int* i, const bool* on, const unsigned long long* stop,
                                          unsigned spin, T* v) {
    using W = ClWord<T>;
    for (unsigned k = 0; k < spin; ++k) {
        typename W::U u[N];
        bool wait = false;
#pragma unroll
        for (int c = 0; c < N; ++c) u[c] = on[c] ? ld_agent((const typename W::U*)hb + i[c]) : 0;
#pragma unroll
        for (int c = 0; c < N; ++c) wait = wait || u[c] == W::empty;
        if (!wait) {
#pragma unroll
            for (int c = 0; c < N; ++c) __builtin_memcpy(&v[c], &u[c], sizeof(T));
            return true;
        }
        if ((k & 63) == 63 && ld_agent(stop) != 0) return false;
    }
    return false;
}

// Neighbour bits (x-, x+, y-, y+, z-, z+) of cell i that the operator sees:
// existing and, with a mask, not behind a masked face.
template <int DIM>
__device__ __forceinline__ int cl_bits_of(const Dims& D, const uint8_t* mask, int i) {
    const int x = i % D.w, t = i / D.w, y = t % D.h, z = t / D.h;
    int has = nbr_bits<DIM>(D, z, y, x);
    if (DIM == 2 && mask) {
        const uint8_t* my = mask;
        const uint8_t* mx = mask + (int64_t)(D.h + 1) * D.w;
        if (!mx[(int64_t)y * (D.w + 1) + x]) has &= ~1;
        if (!mx[(int64_t)y * (D.w + 1) + x + 1]) has &= ~2;
        if (!my[i]) has &= ~4;
        if (!my[i + D.w]) has &= ~8;
    }
    return has;
}

template <typename T, bool JAC>
__device__ __forceinline__ T cl_z(T r, int nc, T dt) {
    if constexpr (JAC) return nc ? r / (dt * (T)nc) : (T)0;
    else return r;
}

__global__ __launch_bounds__(256) void k_cl_reset(ClSlots* s) {
    unsigned long long* w = &s[blockIdx.x].pq[0][0];
    for (int i = threadIdx.x; i < 8 * kClMaxWg; i += 256) w[i] = kClEmpty;
    if (threadIdx.x == 0) s[blockIdx.x].stop = 0;
}

// hb0, hb1: the two copies of the edges of r (n elements each). hb1 may be p:
// it is written first when everybody has read p.
template <typename T, int DIM, int C, int NT, bool JAC>
__global__ __launch_bounds__(NT) void k_cg_cluster(Dims D, int n, int chunk, T* x, T* r, const T* p, T* hb0,
                                                           T* hb1, T dt, const uint8_t* mask, SolverState* st,
                                                           ClSlots* S, unsigned spin) {
    constexpr int NW = NT / 64;
    extern __shared__ __align__(16) char cl_lds[];
    __shared__ double red[2][2][NT / 64];  // sums of the waves: own, then of the slots
    __shared__ int flag;  // cleared when the run is abandoned
    const SolverState s0 = *st;
    if (s0.done) return;
    const int P = gridDim.x, g = blockIdx.x, t = threadIdx.x, wave = t >> 6, mr = g % kClCopies;
    const int w = D.w, hw = D.h * D.w;
    const int f0 = g * chunk, len = imin(chunk, n - f0);
    T* lp = (T*)cl_lds;                            // p of cells [f0 - w, f0 + chunk + w)
    uint8_t* hn = (uint8_t*)(lp + chunk + 2 * w);  // halo cells' diagonal counts (Jacobi)
    const int bc_ = D.bc;
    const int th = NT - 1 - t;  // halo rows start at the last wave: the first ones poll slots

    T xv[C], rv[C], pv[C], zl[C], zh[C];
    int has[C], ncz[C];  // ncz: diagonal counts of the cells above and below (3D Jacobi)
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int o = t + c * NT, i = f0 + o;
        const bool on = o < len;
        xv[c] = (T)0;
        rv[c] = on ? r[i] : (T)0;
        pv[c] = on ? p[i] : (T)0;
        zl[c] = zh[c] = (T)0;
        ncz[c] = 0;
        has[c] = on ? cl_bits_of<DIM>(D, mask, i) : 0;
        if (on && (DIM == 3 || o < w || o >= len - w)) edge_empty(&hb0[i]);
        if (o < chunk) lp[w + o] = pv[c];
        if (DIM == 3 && on) {
            if (has[c] & 16) {
                zl[c] = p[i - hw];
                if (JAC) ncz[c] = ncount_bits<DIM>(cl_bits_of<DIM>(D, mask, i - hw), bc_);
            }
            if (has[c] & 32) {
                zh[c] = p[i + hw];
                if (JAC) ncz[c] |= ncount_bits<DIM>(cl_bits_of<DIM>(D, mask, i + hw), bc_) << 8;
            }
        }
    }
    // halo rows: element e < w is cell f0 - w + e, the others cell f0 + len + e - w
    for (int e = th; e < 2 * w; e += NT) {
        const int i = e < w ? f0 - w + e : f0 + len + e - w;
        const bool on = i >= 0 && i < n;
        lp[e < w ? e : len + e] = on ? p[i] : (T)0;
        if (JAC) hn[e] = on ? (uint8_t)ncount_bits<DIM>(cl_bits_of<DIM>(D, mask, i), bc_) : 0;
    }
    if (t == 0) flag = 1;
    __syncthreads();

    double sigma = s0.sigma, alpha = s0.alpha, beta = s0.beta, pq = s0.pq, rnorm = s0.rnorm;
    int iter = s0.iter, conv = 0, bad = 0;
    // the thread's halo polls behind the exchange's barrier were answered: told
    // at the next exchange, as slower waves may still have to read `flag`
    bool kept = true;
    for (int k = 0; iter < s0.max_iter; ++k) {
        const int k2 = k & 1, k4 = k & 3;
        T* hb = k2 ? hb1 : hb0;
        T* ho = k2 ? hb0 : hb1;
        // q = A p ; alpha (pcg.rs:51-53)
        T q[C];
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int o = t + c * NT, m = w + o;
            q[c] = (T)0;
            if (o < len) {
                q[c] = poisson_from<T, DIM>(pv[c], lp[m - 1], lp[m + 1], lp[m - w], lp[m + w], zl[c], zh[c], has[c],
                                            bc_, dt);
                s += (double)pv[c] * (double)q[c];
            }
        }
        s = wave_all<ClSum>(s);
        if ((t & 63) == 0) red[0][0][wave] = s;
        stores_done();
        __syncthreads();
        if (t < kClCopies) st_agent(&S[t].pq[k4][g], cl_bits(waves_all<ClSum, NW>(red[0][0])));
        double v[2];
        bool got = cl_poll<1>(S[mr].pq[k4], nullptr, &S->stop, P, spin, v);
        s = wave_all<ClSum>(v[0]);
        if ((t & 63) == 0) red[1][0][wave] = s;
        if (!got || !kept) flag = 0;
        __syncthreads();
        if (!flag) break;
        pq = waves_all<ClSum, NW>(red[1][0]);
        alpha = sigma / pq;
        if (!(alpha == alpha) || fabs(alpha) > 1.7e308) {
            bad = 1;
            break;
        }
        // r -= alpha q ; max|r| ; z = M r ; z.r (pcg.rs:55-68)
        double m = 0.0;
        s = 0.0;
        T z[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int o = t + c * NT;
            z[c] = (T)0;
            if (o < len) {
                rv[c] = (T)((double)rv[c] - alpha * (double)q[c]);
                if (DIM == 3 || o < w || o >= len - w) {
                    edge_store(&hb[f0 + o], rv[c]);
                    edge_empty(&ho[f0 + o]);
                }
                m = absmax_acc(m, (double)rv[c]);
                z[c] = cl_z<T, JAC>(rv[c], JAC ? ncount_bits<DIM>(has[c], bc_) : 0, dt);
                s += (double)z[c] * (double)rv[c];
            }
        }
        s = wave_all<ClSum>(s);
        m = wave_all<ClMax>(m);
        if ((t & 63) == 0) {
            red[0][0][wave] = s;
            red[0][1][wave] = m;
        }
        __syncthreads();
        if (t < kClCopies) {
            st_agent(&S[t].zr[k2][g], cl_bits(waves_all<ClSum, NW>(red[0][0])));
            st_agent(&S[t].mx[k2][g], cl_bits(waves_all<ClMax, NW>(red[0][1])));
            // behind the barrier of the p.q exchange, at which the waves together had
            // seen every p.q (a wave has seen its own slots' only), and behind the
            // values that others wait for
            st_agent(&S[t].pq[(k + 3) & 3][g], kClEmpty);
            st_agent(&S[t].zr[k2 ^ 1][g], kClEmpty);
            st_agent(&S[t].mx[k2 ^ 1][g], kClEmpty);
        }
        got = cl_poll<2>(S[mr].zr[k2], S[mr].mx[k2], &S->stop, P, spin, v);
        s = wave_all<ClSum>(v[0]);
        m = wave_all<ClMax>(v[1]);
        if ((t & 63) == 0) {
            red[1][0][wave] = s;
            red[1][1][wave] = m;
        }
        // the neighbours' r at this iteration: z halo into registers, halo rows
        T hz[2 * C];
        if constexpr (DIM == 3) {
            int hi[2 * C];
            bool on[2 * C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int i = f0 + t + c * NT;
                hi[c] = i - hw;
                hi[C + c] = i + hw;
                on[c] = (has[c] & 16) != 0;
                on[C + c] = (has[c] & 32) != 0;
            }
            got = got && edge_poll<T, 2 * C>(hb, hi, on, &S->stop, spin, hz);
        }
        T hr = (T)0;  // the first halo cell of the thread; wider rows' others are polled below
        {
            const int i = th < w ? f0 - w + th : f0 + len + th - w;
            const bool on = th < 2 * w && i >= 0 && i < n;
            got = got && edge_poll<T, 1>(hb, &i, &on, &S->stop, spin, &hr);
        }
        if (!got) flag = 0;
        __syncthreads();
        if (!flag) break;
        rnorm = waves_all<ClMax, NW>(red[1][1]);
        iter += 1;
        // x += alpha p, in both ways out of the iteration
#pragma unroll
        for (int c = 0; c < C; ++c) xv[c] = (T)((double)xv[c] + alpha * (double)pv[c]);
        if (!(rnorm == rnorm)) {
            bad = 1;
            break;
        }
        if (rnorm < s0.threshold) {  // pcg.rs:58-63
            conv = 1;
            break;
        }
        if (iter >= s0.max_iter) break;
        const double zr = waves_all<ClSum, NW>(red[1][0]);
        beta = zr / sigma;
        sigma = zr;
        if (!(beta == beta)) {
            bad = 1;
            break;
        }
        // p = z + beta p (pcg.rs:72-77), here and in the halo
        got = true;
        for (int e = th; e < 2 * w; e += NT) {
            const int i = e < w ? f0 - w + e : f0 + len + e - w, a = e < w ? e : len + e;
            if (i < 0 || i >= n) continue;
            const bool on = true;
            if (e != th) got = got && edge_poll<T, 1>(hb, &i, &on, &S->stop, spin, &hr);
            lp[a] = (T)((double)cl_z<T, JAC>(hr, JAC ? hn[e] : 0, dt) + beta * (double)lp[a]);
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int o = t + c * NT;
            pv[c] = (T)((double)z[c] + beta * (double)pv[c]);
            if (o < len) lp[w + o] = pv[c];
            if constexpr (DIM == 3) {
                zl[c] = (T)((double)cl_z<T, JAC>(hz[c], ncz[c] & 255, dt) + beta * (double)zl[c]);
                zh[c] = (T)((double)cl_z<T, JAC>(hz[C + c], ncz[c] >> 8, dt) + beta * (double)zh[c]);
            }
        }
        kept = got;
        __syncthreads();
    }
    if (!flag) {  // abandoned (uniform): the host starts over with the launches
        if (t == 0) {
            st_agent(&S->stop, 1ull);
            st_agent(&st->stalled, 1);
        }
        return;
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int o = t + c * NT;
        if (o < len) {
            x[f0 + o] = xv[c];
            r[f0 + o] = rv[c];
        }
    }
    if (g == 0 && t == 0) {
        st->sigma = sigma;
        st->alpha = alpha;
        st->beta = beta;
        st->pq = pq;
        st->rnorm = rnorm;
        st->iter = iter;
        st->xit = iter;
        st->converged = conv;
        st->nonfinite = bad;
        st->done = 1;
    }
}

static std::mutex g_cl_mu;
static std::condition_variable g_cl_cv;
static int g_cl_used[64];

ClReserve::ClReserve(int dev, int w, int num_cu) : device(dev & 63), wgs(w) {
    std::unique_lock<std::mutex> lock(g_cl_mu);
    g_cl_cv.wait(lock, [&] { return g_cl_used[device] == 0 || g_cl_used[device] + wgs <= num_cu; });
    g_cl_used[device] += wgs;
}
ClReserve::~ClReserve() {
    {
        std::lock_guard<std::mutex> lock(g_cl_mu);
        g_cl_used[device] -= wgs;
    }
    g_cl_cv.notify_all();
}

// The split. An iteration costs about 3 us of exchange latency plus what its
// cells and its polls take; more workgroups mean fewer cells but more polls.
// Measured at us per iteration (f32 2D unless said; launches: 21 to 33):
// 128^2 4.6 as 64 workgroups of 256 threads, 5.6 as 16 of 1024; 150x203 f64 5.1
// as 60 of 512; 300^2 6.7 as 88 of 1024; 512^2 7.9 as 128 of 1024, two cells
// per thread, 8.2 as 256 of one; 64^3 8.5 as 256 of 1024, 9.1 as 128 (in 3D
// every cell is an edge value, so fewer cells per workgroup win).
ClPlan cl_plan(const Dims& D, size_t elem, int num_cu) {
    ClPlan P;
    const int64_t n = (int64_t)D.d * D.h * D.w;
    const int most = imin(D.d > 1 ? kClMaxWg : kClMaxWg / 2, num_cu);
    if (D.w > kClMaxWidth || n > (int64_t)most * 1024 * kClMaxC) return P;
    P.nt = n <= imin(64, most) * 256 ? 256 : n <= imin(64, most) * 512 ? 512 : 1024;
    P.c = 1;
    while ((int64_t)most * P.nt * P.c < n) P.c *= 2;
    const int per = P.nt * P.c;
    const int wgs = (int)((n + per - 1) / per);
    P.chunk = (int)(((n + wgs - 1) / wgs + 63) / 64 * 64);
    P.lds = (size_t)(P.chunk + 2 * D.w) * elem + 2 * D.w;
    if (P.lds <= (128u << 10)) P.wgs = (int)((n + P.chunk - 1) / P.chunk);
    return P;
}

template <typename T, int DIM, bool JAC>
static void cl_launch(Ctx* c, const Dims& D, const ClPlan& P, T* x, T* r, T* p, T* hb, T dt,
                      const uint8_t* mask, SolverState* st, ClSlots* s, unsigned spin) {
    const int n = D.d * D.h * D.w;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(P.wgs), dim3(P.nt), P.lds, c->stream, D, n, P.chunk, x, r,
                           (const T*)p, hb, p, dt, mask, st, s, spin);
    };
    if (P.nt == 256) go(k_cg_cluster<T, DIM, 1, 256, JAC>);
    else if (P.nt == 512) go(k_cg_cluster<T, DIM, 1, 512, JAC>);
    else if (P.c == 1) go(k_cg_cluster<T, DIM, 1, 1024, JAC>);
    else if (P.c == 2) go(k_cg_cluster<T, DIM, 2, 1024, JAC>);
    else go(k_cg_cluster<T, DIM, 4, 1024, JAC>);
}

template <typename T>
pano_status cl_solve(Ctx* c, const Dims& D, const ClPlan& P, bool jacobi, T* x, T* r, T* p, T* hb, T dt,
                     const uint8_t* mask, SolverState* st, ClSlots* slots, unsigned spin) {
    hipLaunchKernelGGL(k_cl_reset, dim3(kClCopies), dim3(256), 0, c->stream, slots);
    if (D.d > 1) {
        if (jacobi) cl_launch<T, 3, true>(c, D, P, x, r, p, hb, dt, mask, st, slots, spin);
        else cl_launch<T, 3, false>(c, D, P, x, r, p, hb, dt, mask, st, slots, spin);
    } else {
        if (jacobi) cl_launch<T, 2, true>(c, D, P, x, r, p, hb, dt, mask, st, slots, spin);
        else cl_launch<T, 2, false>(c, D, P, x, r, p, hb, dt, mask, st, slots, spin);
    }
    PANO_HIP(hipGetLastError());
    return PANO_OK;
}
template pano_status cl_solve<float>(Ctx*, const Dims&, const ClPlan&, bool, float*, float*, float*, float*, float,
                                     const uint8_t*, SolverState*, ClSlots*, unsigned);
template pano_status cl_solve<double>(Ctx*, const Dims&, const ClPlan&, bool, double*, double*, double*, double*, double,
                                      const uint8_t*, SolverState*, ClSlots*, unsigned);

}  // namespace pano
