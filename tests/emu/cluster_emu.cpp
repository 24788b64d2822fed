// CPU emulation of the one-kernel CG loop (cg_cluster.hip, built from its own
// source with the stand-ins of host_hip/): its workgroups, waves and threads
// run in random order, one wave between two agent-scope loads or barriers at a
// time, stores reach memory out of order and late (at the latest where the
// wave waits for them), and one wave of one workgroup is held back while all
// others go on as far as they can. Whatever the order, the loop has to reach
// its end without a wait running out and give the same bits, for clusters of
// more workgroups than a wave has lanes above all; and where waits run out (a
// few polls allowed only), the waves of a workgroup have to leave together.
#include <sched.h>
#include <semaphore.h>
#include <setjmp.h>
#include <sys/mman.h>
#include <ucontext.h>
#include <unistd.h>

#include <cstdio>
#include <memory>
#include <random>
#include <thread>
#include <vector>

#include "cg_cluster.hip"

thread_local dim3 threadIdx, blockIdx, blockDim, gridDim;
namespace pano {
alignas(16) thread_local char cl_lds[128 << 10];
pano_status fail(pano_status s, const char*, ...) { return s; }
}  // namespace pano
using namespace pano;

// ---- the machine --------------------------------------------------------------------
namespace {

std::mt19937 g_rng(1);
unsigned rnd(unsigned n) { return g_rng() % n; }

enum Lane { RUN, LOAD, COLL, BAR, DONE };
struct Store {
    char* p;
    unsigned char v[8];
    size_t n;
    long due;  // turns of all waves before which it does not arrive by itself
};
long g_turns;
// Late: edge values in these bytes arrive after `turns` only, and wave `wave` of
// workgroup `wg` leaves its `barrier`-th barrier as late.
struct Late {
    const char *lo = nullptr, *hi = nullptr;
    int wg = -1, wave = 0, barrier = 0, turns = 0;
} g_late;
long g_stores;  // that have reached memory
struct Wave {
    Lane st[64];
    jmp_buf at[64];
    bool begun[64];
    int op, in[64], out[64];
    std::vector<Store> pending;
    bool done = false, bar = false;
    int polls = 0;   // scheduling points passed
    int barriers = 0;
    long held = 0;   // turn of all waves up to which this one is held
    int same = 0;    // of them the last ones with no store to memory since
    long seen = -1;
    void flush_one(size_t i, bool wait = false) {
        for (size_t j = 0; j < i; ++j)  // stores to one address stay in order
            if (pending[j].p == pending[i].p) { i = j; break; }
        if (!wait && g_turns < pending[i].due) return;
        ++g_stores;
        memcpy(pending[i].p, pending[i].v, pending[i].n);
        pending.erase(pending.begin() + i);
    }
    void flush() {
        while (!pending.empty()) flush_one(rnd((unsigned)pending.size()), true);
    }
};
constexpr size_t kStack = 24 << 10;
struct Group {
    std::vector<Wave> w;
    char* stacks = nullptr;
    int id = 0, live = 0, pick = 0;
    bool divergent = false;
    sem_t go, back;
    std::thread th;
};
struct Launch {
    dim3 grid, block;
    void (*body)(void*);
    void* arg;
};
thread_local Group* t_g;
thread_local Wave* t_w;
thread_local int t_lane;
thread_local jmp_buf t_sched;
thread_local const Launch* t_l;
bool g_divergent;

// the running lane stops in state s until the scheduler resumes it
void stop(Lane s) {
    Wave* w = t_w;
    const int l = t_lane;
    w->st[l] = s;
    if (_setjmp(w->at[l]) == 0) _longjmp(t_sched, 1);
}
void lane_main() {
    t_l->body(t_l->arg);
    t_w->st[t_lane] = DONE;
    _longjmp(t_sched, 1);
}
void resume(Group* g, int wave, int l) {
    Wave* w = &g->w[wave];
    t_w = w;
    t_lane = l;
    threadIdx = dim3(wave * 64 + l);
    w->st[l] = RUN;
    if (_setjmp(t_sched) != 0) return;
    if (w->begun[l]) _longjmp(w->at[l], 1);
    w->begun[l] = true;
    ucontext_t u;
    getcontext(&u);
    u.uc_stack.ss_sp = g->stacks + (size_t)(wave * 64 + l) * kStack;
    u.uc_stack.ss_size = kStack;
    u.uc_link = nullptr;
    makecontext(&u, lane_main, 0);
    setcontext(&u);
}
// runs one wave up to its next agent-scope load or barrier
void step(Group* g, int wave) {
    Wave& w = g->w[wave];
    for (;;) {
        for (int l = 0; l < 64; ++l)
            if (w.st[l] == RUN || w.st[l] == LOAD) resume(g, wave, l);
        int n[5] = {0, 0, 0, 0, 0};
        for (int l = 0; l < 64; ++l) ++n[w.st[l]];
        if (n[COLL] && !n[LOAD] && !n[BAR]) {
            for (int l = 0; l < 64; ++l) {
                if (w.st[l] != COLL) continue;
                int from = l;
                if (w.op == 1000) {
                    w.out[l] = 0;
                    for (int j = 0; j < 64; ++j) w.out[l] |= w.st[j] == COLL ? w.in[j] : 0;
                    continue;
                }
                if (w.op >= 2000) from = w.op - 2000;
                else if (w.op == 0xB1) from = l ^ 1;
                else if (w.op == 0x4E) from = l ^ 2;
                else if (w.op == 0x141) from = (l & ~7) | (7 - (l & 7));
                else if (w.op == 0x140) from = (l & ~15) | (15 - (l & 15));
                else abort();
                w.out[l] = w.in[from];
            }
            for (int l = 0; l < 64; ++l)
                if (w.st[l] == COLL) w.st[l] = RUN;
            continue;
        }
        if (n[LOAD]) return;
        if (n[DONE] == 64) {
            w.done = true;
            w.flush();
            --g->live;
        } else {
            w.bar = true;
        }
        break;
    }
    int at = 0;
    for (Wave& v : g->w) at += v.bar;
    if (at && at == g->live) {
        if (g->live < (int)g->w.size()) g->divergent = true;  // a wave left, another waits at a barrier
        for (Wave& v : g->w) {
            if (!v.bar) continue;
            v.bar = false;
            v.same = 0;
            if (g->id == g_late.wg && &v == &g->w[g_late.wave] && ++v.barriers == g_late.barrier)
                v.held = g_turns + g_late.turns;
            for (int l = 0; l < 64; ++l)
                if (v.st[l] == BAR) v.st[l] = RUN;
        }
    }
}
int collective(int op, int v) {
    Wave* w = t_w;
    const int l = t_lane;
    w->op = op;
    w->in[l] = v;
    stop(COLL);
    return t_w->out[t_lane];
}

// A wave that polls memory nobody has written to since is left out (unless
// waits are to run out): kIdle polls are more than any loop's loads per try.
// Once that holds for every wave, nothing will ever end the waits.
constexpr int kIdle = 8;
bool g_skip_idle = true;

// The wave to hold back: from its scheduling point `at` on, for `steps` of its turns.
struct Hold {
    int wg = -1, wave = 0, at = 0, steps = 0;
} g_hold;

}  // namespace

void __syncthreads() { stop(BAR); }
bool __any(bool v) { return collective(1000, v) != 0; }
int emu_dpp(int, int v, int ctrl, int, int, bool) { return collective(ctrl, v); }
int emu_readlane(int v, int lane) { return collective(2000 + lane, v); }
void emu_waitcnt() { t_w->flush(); }
void emu_store(void* p, const void* v, size_t n) {
    Store s{(char*)p, {}, n, p >= g_late.lo && p < g_late.hi ? g_turns + g_late.turns : 0};
    memcpy(s.v, v, n);
    t_w->pending.push_back(s);
}
void emu_load(const void* p, void* v, size_t n) {
    stop(LOAD);
    for (size_t i = t_w->pending.size(); i-- > 0;)
        if (t_w->pending[i].p == p) {
            memcpy(v, t_w->pending[i].v, n);
            return;
        }
    memcpy(v, p, n);
}

bool emu_launch(dim3 grid, dim3 block, size_t lds, void (*body)(void*), void* arg) {
    if (lds > sizeof(cl_lds) || block.x % 64) abort();
    const Launch L{grid, block, body, arg};
    std::vector<std::unique_ptr<Group>> gs;
    for (unsigned i = 0; i < grid.x; ++i) {
        gs.emplace_back(new Group);
        Group* g = gs.back().get();
        g->id = i;
        g->w = std::vector<Wave>(block.x / 64);
        g->live = (int)g->w.size();
        for (Wave& w : g->w)
            for (int l = 0; l < 64; ++l) w.st[l] = RUN, w.begun[l] = false;
        g->stacks = (char*)mmap(nullptr, kStack * block.x, PROT_READ | PROT_WRITE,
                                MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (g->stacks == MAP_FAILED) abort();
        sem_init(&g->go, 0, 0);
        sem_init(&g->back, 0, 0);
        g->th = std::thread([g, &L] {
            t_g = g;
            t_l = &L;
            blockIdx = dim3(g->id);
            blockDim = L.block;
            gridDim = L.grid;
            while (true) {
                sem_wait(&g->go);
                if (g->pick < 0) return;
                step(g, g->pick);
                sem_post(&g->back);
            }
        });
    }
    std::vector<std::pair<int, int>> open;  // waves that have not ended
    for (unsigned i = 0; i < grid.x; ++i)
        for (unsigned k = 0; k < block.x / 64; ++k) open.push_back({(int)i, (int)k});
    Hold h = g_hold;
    long idle = 0;
    while (!open.empty()) {
        if (++idle > 100 * (long)open.size()) {
            printf("FAIL no wave can go on: a wait without an end (held: workgroup %d wave %d from point %d)\n", h.wg, h.wave, h.at);
            fflush(stdout);
            _exit(1);
        }
        const unsigned i = rnd((unsigned)open.size());
        ++g_turns;
        Group* g = gs[open[i].first].get();
        const int k = open[i].second;
        Wave& w = g->w[k];
        if (!w.pending.empty()) {
            idle = 0;
            while (!w.pending.empty() && rnd(8)) w.flush_one(rnd((unsigned)w.pending.size()));
        }
        if (w.bar) continue;
        if (g_turns < w.held) {
            idle = 0;
            continue;
        }
        if (g->id == h.wg && k == h.wave && w.polls >= h.at && h.steps > 0) {
            --h.steps;
            idle = 0;
            continue;
        }
        w.same = w.seen == g_stores ? w.same + 1 : 0;
        w.seen = g_stores;
        if (g_skip_idle && w.same > kIdle) continue;
        idle = 0;
        ++w.polls;
        g->pick = k;
        sem_post(&g->go);
        sem_wait(&g->back);
        if (w.done) {
            open[i] = open.back();
            open.pop_back();
        }
    }
    for (auto& g : gs) {
        g->pick = -1;
        sem_post(&g->go);
        g->th.join();
        munmap(g->stacks, kStack * block.x);
        g_divergent = g_divergent || g->divergent;
    }
    return true;
}

// ---- the solves ---------------------------------------------------------------------
template <typename T>
struct Run {
    std::vector<T> x, r;
    SolverState st;
    bool operator==(const Run& o) const {
        return memcmp(x.data(), o.x.data(), x.size() * sizeof(T)) == 0 &&
               memcmp(r.data(), o.r.data(), r.size() * sizeof(T)) == 0 && memcmp(&st, &o.st, sizeof(st)) == 0;
    }
};

template <typename T>
static Run<T> solve(const Dims& D, int chunk, bool jacobi, int iterations, unsigned spin) {
    const int n = D.d * D.h * D.w;
    std::mt19937 rng(7);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    Run<T> R;
    R.x.assign(n, (T)0);
    R.r.resize(n);
    std::vector<T> p(n), hb(n);
    const T dt = (T)0.3;
    memset(&R.st, 0, sizeof(R.st));
    for (int i = 0; i < n; ++i) {
        R.r[i] = (T)U(rng);
        const int bits = D.d > 1 ? cl_bits_of<3>(D, nullptr, i) : cl_bits_of<2>(D, nullptr, i);
        const int nc = D.d > 1 ? ncount_bits<3>(bits, D.bc) : ncount_bits<2>(bits, D.bc);
        p[i] = jacobi ? cl_z<T, true>(R.r[i], nc, dt) : R.r[i];
        R.st.sigma += (double)p[i] * (double)R.r[i];
    }
    R.st.max_iter = iterations;
    ClPlan P;
    P.nt = 256;
    P.c = 1;
    P.chunk = chunk;
    P.wgs = (n + chunk - 1) / chunk;
    P.lds = (size_t)(chunk + 2 * D.w) * sizeof(T) + 2 * D.w;
    static ClSlots slots[kClCopies];
    const int behind = (g_late.wg + 1) * chunk;
    g_late.lo = g_late.wg < 0 ? nullptr : (const char*)(hb.data() + behind);
    g_late.hi = g_late.wg < 0 ? nullptr : (const char*)(hb.data() + (behind + 100 < n ? behind + 100 : n));
    Ctx c;
    cl_solve<T>(&c, D, P, jacobi, R.x.data(), R.r.data(), p.data(), hb.data(), dt, nullptr, &R.st, slots, spin);
    return R;
}

static int fails = 0, runs = 0;

template <typename T>
static void orders(const char* what, const Dims& D, int chunk, bool jacobi, int iterations, int seeds) {
    const int wgs = (D.d * D.h * D.w + chunk - 1) / chunk;
    const unsigned spin = 1u << 30;  // an order with no end is found by the scheduler
    g_rng.seed(1);
    g_hold = Hold();
    g_divergent = false;
    const Run<T> ref = solve<T>(D, chunk, jacobi, iterations, spin);
    for (int s = 0; s <= seeds; ++s) {
        if (s > 0) {
            g_rng.seed(100 + s);
            // most often a workgroup whose slot is not the first wave's, anywhere in the run
            g_hold.wg = wgs > 64 && s % 4 ? 64 + (int)rnd(wgs - 64) : (int)rnd(wgs);
            g_hold.wave = (int)rnd(s % 2 ? 1 : 4);
            g_hold.at = (int)rnd(10 * iterations);
            g_hold.steps = 400;
        }
        const Run<T> R = s ? solve<T>(D, chunk, jacobi, iterations, spin) : ref;
        ++runs;
        const bool ok = !R.st.stalled && R.st.done && R.st.iter == iterations && R == ref && !g_divergent;
        if (!ok) {
            ++fails;
            printf("FAIL %s %d workgroups, order %d (held: workgroup %d wave %d): stalled %d done %d iterations %d "
                   "same %d\n", what, wgs, s, g_hold.wg, g_hold.wave, R.st.stalled, R.st.done, R.st.iter,
                   (int)(R == ref));
            fflush(stdout);
            return;
        }
    }
}

// Waits run out after `spin` polls: an abandoned run says so, and no wave waits
// at a barrier for one that has left.
template <typename T>
static void abandoned(const char* what, const Dims& D, int chunk, int iterations, int seeds) {
    g_skip_idle = false;
    g_hold = Hold();
    int stalls = 0;
    for (int s = 0; s < seeds; ++s) {
        g_rng.seed(1000 + s);
        g_divergent = false;
        const unsigned spin = 30 + rnd(120);
        // the first cells behind a workgroup's own, which long rows poll behind the exchange's barrier
        g_late.wg = (int)rnd(D.d * D.h * D.w / chunk - 1);
        g_late.wave = (int)rnd(4);
        g_late.barrier = 1 + (int)rnd(6);
        g_late.turns = 30000;
        const Run<T> R = solve<T>(D, chunk, true, iterations, spin);
        ++runs;
        stalls += R.st.stalled != 0;
        if (g_divergent || !(R.st.stalled || (R.st.done && R.st.iter == iterations))) {
            ++fails;
            printf("FAIL %s, order %d, %u polls: %s stalled %d done %d\n", what, s, spin,
                   g_divergent ? "a wave left its workgroup's others at a barrier" : "", R.st.stalled, R.st.done);
        }
    }
    printf("%s: %d of %d runs abandoned\n", what, stalls, seeds);
    g_skip_idle = true;
    g_late = Late();
}

// Solves of a context whose loops are all given up, then end again.
static void use() {
    ClusterUse u;
    std::string seen;
    for (int k = 0; k < 40; ++k) {
        const bool t = u.take();
        seen += t ? 'x' : '.';
        if (t) u.ended(true);
    }
    int longest = 0, run = 0;
    for (int k = 0; k < 10000; ++k) {
        const bool t = u.take();
        run = t ? 0 : run + 1;
        longest = run > longest ? run : longest;
        if (t) u.ended(true);
    }
    while (!u.take()) {
    }
    u.ended(false);
    bool back = u.take();
    u.ended(true);  // the first one again: no solve is left out
    back = back && u.take();
    ++runs;
    if (seen != "xx.x...x.......x...............x........" || longest != 1023 || !back) {
        ++fails;
        printf("FAIL the solves that stay with the launches: %s, %d at most, back %d\n", seen.c_str(), longest, back);
    }
}

int main() {
    cpu_set_t one;  // one thread runs at a time
    CPU_ZERO(&one);
    CPU_SET(sched_getcpu(), &one);
    sched_setaffinity(0, sizeof(one), &one);
    orders<float>("2D identity", Dims{1, 66, 64, 0}, 64, false, 4, 4);
    orders<float>("2D Jacobi, rows wider than a workgroup's cells", Dims{1, 15, 300, 1}, 64, true, 4, 3);
    orders<double>("3D Jacobi", Dims{17, 16, 17, 32}, 64, true, 4, 3);
    orders<double>("2D identity", Dims{1, 130, 64, 2}, 64, false, 3, 2);
    orders<float>("2D identity", Dims{1, 256, 64, 0}, 64, false, 2, 1);
    use();
    abandoned<float>("few workgroups, long rows", Dims{1, 3, 300, 0}, 64, 3, 60);
    printf("%d orders, %d failures\n", runs, fails);
    return fails != 0;
}
