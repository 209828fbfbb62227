// What a handle does when memory cannot be had, and a rollout's two layouts,
// on the GPU.  The program stands between the library and the runtime: it can
// make a device or pinned allocation fail (by asking the runtime for
// more than there is, so that the runtime records its error), and it can say
// that no device memory is free, which leaves a rollout with the caller's
// checkpoints.  Prints one line per check and returns how many failed.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>

#include <hip/hip_runtime.h>

#include "opencloth.h"

namespace {
int g_fail_device = 0, g_fail_pinned = 0;  // n: the n-th from here
bool g_no_memory = false;
int g_asked = 0, g_wrong = 0;

template <class F>
F real(const char* name) {
    F f = (F)dlsym(RTLD_NEXT, name);
    if (!f) std::printf("no %s\n", name), std::fflush(stdout);
    return f;
}
void check(const char* what, int a, int b, bool ok) {
    std::printf("%s %d %d %s\n", what, a, b, ok ? "ok" : "WRONG");
    std::fflush(stdout);
    g_wrong += !ok;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    static const auto f = real<hipError_t (*)(void**, size_t)>("hipMalloc");
    if (g_fail_device && --g_fail_device == 0) n = size_t(1) << 50;
    return f(p, n);
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    static const auto f = real<hipError_t (*)(void**, size_t, unsigned)>("hipHostMalloc");
    if (g_fail_pinned && --g_fail_pinned == 0) n = size_t(1) << 50;
    return f(p, n, flags);
}
hipError_t hipMemGetInfo(size_t* avail, size_t* total) {
    static const auto f = real<hipError_t (*)(size_t*, size_t*)>("hipMemGetInfo");
    const hipError_t e = f(avail, total);
    g_asked++;
    if (g_no_memory) *avail = 0;
    return e;
}
}

static const int kNx = 40, kNy = 30, kN = kNx * kNy;
static std::vector<float> g_x(3 * kN), g_v(3 * kN, 0.0f), g_grad(3 * kN);
static std::vector<oc_spring> g_springs;
static std::vector<uint8_t> g_pins(kN, 0);

static void scene() {
    unsigned h = 1;
    auto rnd = [&]() { return (float)((h = h * 1664525u + 1013904223u) >> 8) / 16777216.0f - 0.5f; };
    for (int k = 0; k < kN; k++) {
        g_x[3 * k] = 0.1f * (k % kNx) + 0.001f * rnd();
        g_x[3 * k + 1] = 0.001f * rnd();
        g_x[3 * k + 2] = 0.1f * (k / kNx) + 0.001f * rnd();
        for (int c = 0; c < 3; c++) g_grad[3 * k + c] = rnd();
    }
    auto add = [](int a, int b, float l) { g_springs.push_back({a, b, l, 50.0f, -0.25f, 0}); };
    for (int j = 0; j < kNy; j++)
        for (int i = 0; i + 1 < kNx; i++) add(j * kNx + i, j * kNx + i + 1, 0.1f);
    for (int j = 0; j + 1 < kNy; j++)
        for (int i = 0; i < kNx; i++) add(j * kNx + i, (j + 1) * kNx + i, 0.1f);
    for (int i = 0; i < kNx; i++) g_pins[i] = 1;
}

static oc_params params() {
    oc_params p = {};
    p.mass = 1.0f;
    p.gravity[1] = -9.81f;
    p.dt = 1.0f / 60.0f;
    p.cg_max_iters = 12;
    p.cg_tol_mode = 2;
    return p;
}

// A cloth (batch: of two), its rollout and its gradients.
struct Run {
    oc_cloth c = nullptr;
    oc_batch b = nullptr;
    size_t copies;
    explicit Run(bool batch) : copies(batch ? 2 : 1) {
        const oc_params p = params();
        if (!batch) {
            if (oc_cloth_create(kNx, kNy, g_x.data(), g_v.data(), g_springs.data(), (int)g_springs.size(),
                                g_pins.data(), &p, &c) != OC_OK)
                c = nullptr;
            return;
        }
        const int32_t nx[2] = {kNx, kNx}, ny[2] = {kNy, kNy}, ns[2] = {(int)g_springs.size(), (int)g_springs.size()};
        std::vector<float> x(g_x), v(g_v);
        std::vector<oc_spring> sp(g_springs);
        std::vector<uint8_t> pins(g_pins);
        x.insert(x.end(), g_x.begin(), g_x.end());
        v.insert(v.end(), g_v.begin(), g_v.end());
        sp.insert(sp.end(), g_springs.begin(), g_springs.end());
        pins.insert(pins.end(), g_pins.begin(), g_pins.end());
        if (oc_batch_create(2, nx, ny, x.data(), v.data(), sp.data(), ns, pins.data(), &p, &b) != OC_OK) b = nullptr;
    }
    ~Run() {
        if (c) oc_cloth_destroy(c);
        if (b) oc_batch_destroy(b);
    }
    bool made() const { return c || b; }
    bool start() {
        std::vector<float> x, v;
        for (size_t k = 0; k < copies; k++) {
            x.insert(x.end(), g_x.begin(), g_x.end());
            v.insert(v.end(), g_v.begin(), g_v.end());
        }
        return (c ? oc_cloth_set_state(c, x.data(), v.data()) : oc_batch_set_state(b, x.data(), v.data())) == OC_OK;
    }
    bool gradients(int steps, int every, std::vector<float>& out) {
        const size_t n = 3 * kN * copies, s = g_springs.size() * copies;
        std::vector<float> g;
        for (size_t k = 0; k < copies; k++) g.insert(g.end(), g_grad.begin(), g_grad.end());
        out.assign(s + 2 * n, 0.0f);
        float* const ks = out.data();
        if (!start()) return false;
        if (c)
            return oc_cloth_rollout_forward(c, steps, every) == OC_OK &&
                   oc_cloth_rollout_backward(c, g.data(), nullptr, ks, ks + s, ks + s + n) == OC_OK;
        return oc_batch_rollout_forward(b, steps, every) == OC_OK &&
               oc_batch_rollout_backward(b, g.data(), nullptr, ks, ks + s, ks + s + n) == OC_OK;
    }
};

static bool same(const std::vector<float>& a, const std::vector<float>& b) {
    return a.size() == b.size() && std::memcmp(a.data(), b.data(), a.size() * sizeof(float)) == 0;
}

int main() {
    scene();
    const int grid[][2] = {{1, 1}, {5, 2}, {6, 3}, {7, 7}, {9, 4}};
    for (int batch = 0; batch < 2; batch++) {
        for (const auto& g : grid) {
            std::vector<float> all, few, grown, failed;
            Run a(batch), b(batch);
            const int before = g_asked;
            bool ok = a.made() && b.made() && a.gradients(g[0], g[1], all) && g_asked > before;
            g_no_memory = true;  // the caller's checkpoints
            const int mid = g_asked;
            ok = ok && b.gradients(g[0], g[1], few) && g_asked > mid;
            g_no_memory = false;
            check(batch ? "batch: checkpoints" : "cloth: checkpoints", g[0], g[1], ok && same(all, few));
            // the same arena for a rollout that keeps every state, and checkpoints in one that did
            ok = b.gradients(g[0] + 5, g[1], grown) && b.gradients(g[0], g[1], grown);
            check(batch ? "batch: grown" : "cloth: grown", g[0], g[1], ok && same(all, grown));
            g_no_memory = true;
            ok = a.gradients(g[0] + 5, g[1], few) && a.gradients(g[0], g[1], few);
            g_no_memory = false;
            check(batch ? "batch: back" : "cloth: back", g[0], g[1], ok && same(all, few));
            if (g[1] > 1) {  // no memory for every state: the rollout goes on with checkpoints
                Run d(batch);
                ok = d.made();
                g_fail_device = 1;
                ok = ok && d.gradients(g[0], g[1], failed) && g_fail_device == 0;
                check(batch ? "batch: failed" : "cloth: failed", g[0], g[1], ok && same(all, failed));
            }
        }
        // a handle that cannot be made leaves nothing behind for another one
        std::vector<float> first, after;
        Run e(batch);
        bool ok = e.made() && e.gradients(4, 2, first);
        g_fail_device = 1;
        Run none(batch);
        ok = ok && !none.made() && g_fail_device == 0 && e.gradients(4, 2, after);
        check(batch ? "batch: create fails" : "cloth: create fails", 0, 0, ok && same(first, after));
    }
    {  // pinned memory that is not there when a handle is made is asked for again
        oc_verlet_params vp = {};
        vp.mass = 1.0f;
        vp.dt = 1.0f / 60.0f;
        vp.damping = -0.0125f;
        std::vector<float> x[3], xl[3];
        for (int k = 0; k < 3; k++) {  // none, the error word, the transfers'
            oc_verlet v = nullptr;
            x[k].resize(3 * kN);
            xl[k].resize(3 * kN);
            g_fail_pinned = k;
            bool ok = oc_verlet_create(kNx, kNy, g_x.data(), nullptr, g_springs.data(), (int)g_springs.size(),
                                       g_pins.data(), &vp, &v) == OC_OK;
            ok = ok && g_fail_pinned == 0 && oc_verlet_step(v, 3, nullptr) == OC_OK &&
                 oc_verlet_step(v, 6, nullptr) == OC_OK && oc_verlet_get_state(v, x[k].data(), xl[k].data()) == OC_OK;
            check("verlet: pinned memory", k, 0, ok && same(x[k], x[0]) && same(xl[k], xl[0]));
            if (v) oc_verlet_destroy(v);
        }
        oc_batch b = nullptr;
        const oc_params p = params();
        const int32_t nx = kNx, ny = kNy, ns = (int)g_springs.size();
        g_fail_pinned = 1;  // the transfers' slots
        bool ok = oc_batch_create(1, &nx, &ny, g_x.data(), nullptr, g_springs.data(), &ns, g_pins.data(), &p, &b) == OC_OK;
        ok = ok && g_fail_pinned == 0 && oc_batch_step(b, 2) == OC_OK && oc_batch_synchronize(b) == OC_OK;
        check("batch: pinned memory", 0, 0, ok);
        if (b) oc_batch_destroy(b);
    }
    std::printf("wrong %d\n", g_wrong);
    return g_wrong;
}
