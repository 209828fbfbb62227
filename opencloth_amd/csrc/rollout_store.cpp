// Device memory of differentiable rollouts.
#include <algorithm>

#include "oc_internal.hpp"

namespace oc {

// Keeping every state saves the backward pass the second run of every step
// (a third of a 128x128 rollout's time); it takes 36 bytes per vertex and
// step.  The caller's checkpoint_every says how much memory a rollout may
// take, so every state is kept only where that is at most kTimes of it (with
// checkpoints every sqrt(n) steps: rollouts of up to some 250 steps), and
// beyond that at most one kShare-th of the free memory and kMost.
constexpr size_t kTimes = 8, kShare = 8, kMost = size_t(8) << 30;

hipError_t RolloutStore::reserve(size_t n, int nsteps, int checkpoint_every, size_t tail, hipStream_t st) {
    steps = nsteps;
    every = std::min(checkpoint_every, nsteps);
    auto need = [&](bool with_all) {
        all = with_all;
        return sizeof(float) * (3 * kept_floats(n) * ((size_t)states() + every) + tail);
    };
    const size_t least = need(false);
    size_t want = need(true);
    if (want <= bytes) return hipSuccess;
    bool fits = want / kTimes <= least;
    if (fits && least <= bytes) {  // only to grow: not while the stream's work is captured
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        fits = hip_ok(hipStreamIsCapturing(st, &cap)) && cap == hipStreamCaptureStatusNone;
    }
    if (fits) {
        size_t avail = 0, total = 0;
        fits = hip_ok(hipMemGetInfo(&avail, &total)) && want <= std::min(avail / kShare, kMost);
    }
    if (!fits) want = need(false);
    if (want <= bytes) return hipSuccess;
    void* fresh = nullptr;
    if (all && !hip_ok(hipMalloc(&fresh, want))) {
        fresh = nullptr;
        want = need(false);
        if (want <= bytes) return hipSuccess;
    }
    if (arena) {
        const hipError_t r = hipStreamSynchronize(st);
        if (r != hipSuccess) {
            if (fresh) (void)hipFree(fresh);
            return r;
        }
        (void)hipFree(arena);
        arena = nullptr;
        bytes = 0;
    }
    if (!fresh) {
        const hipError_t r = hipMalloc(&fresh, want);
        if (r != hipSuccess) return r;
    }
    arena = fresh;
    bytes = want;
    return hipSuccess;
}

}  // namespace oc
