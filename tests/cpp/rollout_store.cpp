// The rollout store (rollout_store.cpp) over a stand-in for the HIP runtime:
// a device with so much free memory, an allocator that can be told to fail,
// and a last error that stays until it is taken, as the runtime's does.
// Prints one line per check and returns the number of those that failed.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "oc_internal.hpp"

namespace {
size_t g_free = size_t(256) << 30;  // what hipMemGetInfo says
size_t g_most = ~size_t(0);         // larger allocations fail
bool g_info_fails = false, g_capturing = false;
hipError_t g_last = hipSuccess;
size_t g_bytes = 0;  // of the last allocation
int g_live = 0, g_wrong = 0;
char g_arena[1];

hipError_t note(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}
void check(const char* what, long a, long b, bool ok) {
    std::printf("%s %ld %ld %s\n", what, a, b, ok ? "ok" : "WRONG");
    g_wrong += !ok;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_most) return note(hipErrorOutOfMemory);
    g_bytes = n;
    g_live++;
    *p = g_arena;
    return hipSuccess;
}
hipError_t hipFree(void*) { return g_live--, hipSuccess; }
hipError_t hipMemGetInfo(size_t* avail, size_t* total) {
    if (g_info_fails) return note(hipErrorInvalidValue);
    *avail = *total = g_free;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
}

// Kept steps, segments and the rest lie apart, in order, inside the arena.
static bool laid_out(const oc::RolloutStore& r, size_t n, size_t tail) {
    const size_t one = 3 * oc::kept_floats(n) * sizeof(float);
    std::set<const char*> at;
    int kept = 0;
    for (int k = 0; k <= r.steps; k++)
        if (r.keeps(k)) at.insert((const char*)r.state(n, k)), kept++;
    for (int k = 0; k < r.every; k++) at.insert((const char*)r.segment(n, k));
    if ((int)at.size() != kept + r.every || kept != r.states()) return false;
    const char* p = (const char*)r.arena;
    for (const char* q : at) {
        if (q != p) return false;
        p += one;
    }
    return (const char*)r.rest(n) == p && (size_t)(p - (const char*)r.arena) + tail * sizeof(float) <= r.bytes;
}

int main() {
    const size_t n = 1000, tail = 7000;
    const int grid[][2] = {{1, 1}, {1, 5}, {5, 1}, {5, 2}, {6, 3}, {7, 7}, {4, 9}, {24, 8}, {23, 5}};
    for (const auto& g : grid) {
        oc::RolloutStore all, few;
        g_free = size_t(256) << 30;
        bool ok = all.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && all.all && laid_out(all, n, tail);
        check("every state", g[0], g[1], ok);
        g_free = 0;
        ok = few.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && !few.all && laid_out(few, n, tail) &&
             few.bytes <= all.bytes;
        check("checkpoints", g[0], g[1], ok);
        const size_t least = few.bytes;
        // an arena that held one layout takes the other and a shorter rollout
        ok = all.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && all.all && laid_out(all, n, tail);
        check("arena kept", g[0], g[1], ok);
        g_free = size_t(256) << 30;
        ok = few.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && few.all && laid_out(few, n, tail);
        check("arena grown", g[0], g[1], ok);
        // no memory for every state: the caller's checkpoints, and no error left behind
        oc::RolloutStore tight;
        g_most = all.bytes - 1;
        const hipError_t e = tight.reserve(n, g[0], g[1], tail, nullptr);
        ok = least > g_most ? e == hipErrorOutOfMemory  // (they are the same states)
                            : e == hipSuccess && !tight.all && laid_out(tight, n, tail) && g_last == hipSuccess;
        check("allocation failed", g[0], g[1], ok);
        g_most = ~size_t(0);
        g_last = hipSuccess;
        oc::RolloutStore blind;
        g_info_fails = true;
        ok = blind.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && !blind.all && laid_out(blind, n, tail) &&
             g_last == hipSuccess;
        check("free memory not known", g[0], g[1], ok);
        g_info_fails = false;
        g_last = hipSuccess;
        // while captured: what there is, without growing
        g_capturing = true;
        const size_t before = blind.bytes;
        ok = blind.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && laid_out(blind, n, tail) && blind.bytes == before;
        check("captured", g[0], g[1], ok);
        g_capturing = false;
    }
    // the caller's checkpoint_every bounds the memory, however much is free
    const int lengths[][2] = {{24, 8}, {120, 10}, {400, 20}, {1000, 32}, {5000, 70}, {5000, 1}, {5000, 5000}};
    for (const auto& g : lengths) {
        oc::RolloutStore r, few;
        g_free = 0;
        bool ok = few.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess;
        g_free = ~size_t(0) / 2;
        ok = ok && r.reserve(n, g[0], g[1], tail, nullptr) == hipSuccess && laid_out(r, n, tail) &&
             r.bytes <= 8 * few.bytes && (r.all || (size_t)(g[0] + 1) * 9 * oc::kept_floats(n) > 7 * few.bytes / 4);
        check("bounded by the checkpoints", g[0], g[1], ok);
    }
    // no room at all: the error goes to the caller
    oc::RolloutStore none;
    g_most = 0;
    check("no room", 0, 0, none.reserve(n, 4, 2, tail, nullptr) == hipErrorOutOfMemory && !none.arena);
    return g_wrong;
}
