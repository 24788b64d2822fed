// The whole CG loop of a small natural-layout solve (identity or Jacobi) as
// one kernel: a cluster of at most 256 workgroups that keeps x, r and p on the
// chip and exchanges two sums and the residual's edges per iteration.
#pragma once

#include "fluid_device.hpp"
#include "solver_device.hpp"

namespace pano {

constexpr int kClMaxWg = 256;      // each thread of a workgroup polls one slot
constexpr int kClMaxC = 4;         // cells per thread
constexpr int kClCopies = 8;       // mailboxes, one per XCD
constexpr unsigned kClSpin = 1u << 18;  // polls (about 1 us each) before a run is abandoned
constexpr int kClMaxWidth = 2048;  // rows wider than this take the launches

// One mailbox: p.q, z.r and max|r| of every workgroup, in copies taken in
// turn, and the stop word of an abandoned run.
struct ClSlots {
    unsigned long long pq[4][kClMaxWg], zr[2][kClMaxWg], mx[2][kClMaxWg], stop, pad[31];
};

struct ClPlan {
    int wgs = 0;    // 0: the solve takes the launches
    int nt = 256;   // threads per workgroup
    int c = 1;      // cells per thread
    int chunk = 0;  // consecutive cells per workgroup
    size_t lds = 0;
};

// The cluster's split of a solve on a device of num_cu CUs.
ClPlan cl_plan(const Dims& D, size_t elem, int num_cu = kClMaxWg);

// A cluster's share of its device's CUs, from before its launch until it has
// ended: clusters of several contexts that would not fit together wait here
// for each other (on the device they would wait for workgroups that cannot start).
struct ClReserve {
    ClReserve(int device, int wgs, int num_cu);
    ~ClReserve();
    ClReserve(const ClReserve&) = delete;
    ClReserve& operator=(const ClReserve&) = delete;

private:
    int device, wgs;
};

// Runs the loop from the state that solver_init left (r, p, sigma, threshold;
// x = 0) and writes x, r and the final state. p and hb (n elements) are
// overwritten.
// spin: polls of one exchange before the run is abandoned (SolverState::stalled).
template <typename T>
pano_status cl_solve(Ctx* c, const Dims& D, const ClPlan& P, bool jacobi, T* x, T* r, T* p, T* hb, T dt,
                     const uint8_t* mask, SolverState* st, ClSlots* slots, unsigned spin);

}  // namespace pano
