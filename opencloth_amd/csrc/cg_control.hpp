// Control words of an implicit cloth's solves: taking a solve's iteration
// count and status, and preparing the next one.  Device code; it needs
// partial_sum (oc_device.hpp) before it, or a host stand-in that also brings
// threadIdx, __syncthreads and atomicOr.
#pragma once

#include "oc_internal.hpp"

namespace oc {
namespace dev {

// Iteration count and status of the solve, by all threads of one block
// (uniform control flow: partial_sum synchronises the block).  Bits are
// OR-ed in, so update blocks may flag non-finite values concurrently.
__device__ inline void cg_finish_block(const DevCloth& c, const StepScalars& s, float* bc) {
    const int done = c.ctl[0];
    int it;
    float delta;
    if (done) {
        it = c.ctl[1];
        delta = c.scal[it];
    } else {
        it = s.max_it;
        delta = partial_sum(c.del_part + (size_t)it * c.nt, c.nt, bc);
    }
    // r0.r0: written by the first spmv phase, or equal to delta without iterations
    const float delta0 = s.max_it > 0 ? c.scal[0] : delta;
    if (threadIdx.x == 0) {
        const float thresh = s.tol_mode == 1 ? s.tol2 * delta0 : s.tol2;
        const int st = c.ctl[2];
        int extra = 0;
        if (s.tol_mode != 2 && delta > thresh && !(st & OC_SOLVE_BREAKDOWN))
            extra |= OC_SOLVE_NOT_CONVERGED;
        if (!isfinite(delta)) extra |= OC_SOLVE_NONFINITE;
        c.ctl[1] = it;
        atomicOr(c.ctl + 2, extra);
        atomicOr(c.ctl + 3, st | extra);
    }
}

// Control words of the solve that follows an assembly (one thread): not done,
// no status; for the resident solve a new roll call, new tickets and the
// epoch base (past every tag the last resident solve used).
__device__ inline void start_solve(const DevCloth& c) {
    c.ctl[0] = 0;
    c.ctl[1] = 0;
    c.ctl[2] = 0;
    if (c.res_vt) {
        c.sync[0] = c.sync[3];
        c.sync[1] = 0;
        c.sync[kSyncTickets] = c.sync[kSyncTickets + kTicketDone] = 0;
    }
}

// Both, by all threads of one block of an assembly.  AFTER_SOLVE: no launch
// has recorded the previous solve's count and status yet (its update is part
// of this assembly), so they go into the sticky word first.  Every thread has
// read the words, and with them which way through cg_finish_block it takes,
// before one clears them: only one of the ways has a barrier.
template <bool AFTER_SOLVE>
__device__ inline void begin_solve(const DevCloth& c, const StepScalars& s, float* bc) {
    if (AFTER_SOLVE) {
        cg_finish_block(c, s, bc);
        __syncthreads();
    }
    if (threadIdx.x == 0) start_solve(c);
}

}  // namespace dev
}  // namespace oc
