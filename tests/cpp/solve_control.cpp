// An assembly's control words (cg_control.hpp) run on the host by the threads
// of one block, in an order the device allows: thread 0 goes first, as far as
// its next barrier, and only then the others start.  Whatever the previous
// solve left, every thread has to pass the same barriers (a wave that passes
// one more pairs it with the kernel's next), and the count, the status and the
// next solve's words have to be right.  Prints per case: the barriers of
// thread 0, how many threads passed others, and whether the words are right.
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

#include "oc_internal.hpp"

namespace {

constexpr int kThreads = 8;

struct Index {
    int x;
};
thread_local Index threadIdx;

// A barrier that also lets go when every other thread has finished, so that a
// thread which passes one barrier more than the others ends all the same.
std::mutex g_lock;
std::condition_variable g_change;
int g_passed[kThreads];
bool g_waits[kThreads], g_done[kThreads];

bool all_here(int n) {  // every thread has reached barrier n, or is done
    for (int t = 0; t < kThreads; t++)
        if (!g_done[t] && g_passed[t] + (g_waits[t] ? 1 : 0) < n) return false;
    return true;
}

void __syncthreads() {
    std::unique_lock<std::mutex> hold(g_lock);
    const int t = threadIdx.x, n = g_passed[t] + 1;
    g_waits[t] = true;
    g_change.notify_all();
    g_change.wait(hold, [&] { return all_here(n); });
    g_passed[t] = n;
    g_waits[t] = false;
    g_change.notify_all();
}

int atomicOr(int* p, int v) { return __atomic_fetch_or(p, v, __ATOMIC_RELAXED); }

}  // namespace

namespace oc {
namespace dev {
using std::isfinite;
inline float partial_sum(const float* part, int nt, float* bc) {
    if (threadIdx.x == 0) {
        *bc = 0.0f;
        for (int k = 0; k < nt; k++) *bc += part[k];
    }
    __syncthreads();
    return *bc;
}
}  // namespace dev
}  // namespace oc

#include "cg_control.hpp"

int main() {
    for (int done = 0; done < 2; done++)
        for (int res = 0; res < 2; res++) {
            constexpr int its = 3, nt = 5;
            int ctl[8] = {done, done ? 2 : 0, 0, 0, 0, 0, 0, 0};
            float scal[2 * (its + 2)] = {9.0f, 4.0f, 1.0f, 0.0f}, part[(its + 1) * nt] = {};
            for (int k = 0; k < nt; k++) part[its * nt + k] = 0.5f;
            unsigned sync[oc::kSyncWords] = {100u, 7u, 7u, 160u};
            oc::DevCloth c;
            std::memset((void*)&c, 0, sizeof(c));
            c.nt = nt;
            c.ctl = ctl;
            c.scal = scal;
            c.del_part = part;
            c.sync = sync;
            c.res_vt = res;
            oc::StepScalars s{};
            s.max_it = its;
            s.tol_mode = 0;
            s.tol2 = 2.0f;  // left over: 1 after 2 iterations (met), 2.5 after all of them (not met)
            for (int t = 0; t < kThreads; t++) {
                g_passed[t] = 0;
                g_waits[t] = g_done[t] = false;
            }
            float bc = 0.0f;
            std::vector<std::thread> th;
            for (int t = 0; t < kThreads; t++)
                th.emplace_back([&, t] {
                    threadIdx.x = t;
                    if (t > 0) {
                        std::unique_lock<std::mutex> hold(g_lock);
                        g_change.wait(hold, [&] { return g_waits[0] || g_done[0] || g_passed[0] > 0; });
                    }
                    oc::dev::begin_solve<true>(c, s, &bc);
                    const std::lock_guard<std::mutex> hold(g_lock);
                    g_done[t] = true;
                    g_change.notify_all();
                });
            for (std::thread& t : th) t.join();
            int other = 0;
            for (int t = 1; t < kThreads; t++) other += g_passed[t] != g_passed[0];
            const int status = done ? 0 : OC_SOLVE_NOT_CONVERGED;
            const bool right = ctl[0] == 0 && ctl[1] == 0 && ctl[2] == 0 && ctl[3] == status &&
                               (!res || (sync[0] == 160u && sync[1] == 0u && sync[oc::kSyncTickets] == 0u));
            std::printf("done %d resident %d: %d %d %d\n", done, res, g_passed[0], other, right ? 1 : 0);
        }
    return 0;
}
