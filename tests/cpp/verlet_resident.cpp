// The resident Verlet steps from inside, on the GPU.  argv[1]: what to run.
//   launches: a call of many steps is split over launches of bounded length,
//             with the same bits as shorter calls (the program counts the
//             library's launches on their way to the runtime)
//   teams:    steps of resident launches against single steps, with every
//             block and with fewer than there are regions, so that the roll
//             never fills and the steps are done by tickets
//   lost:     after a wait between blocks that ended without its word (the
//             program sets the error word itself), every call that uses the
//             state says so until the caller has given a new one
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "oc_internal.hpp"

namespace {
int g_launches = 0, g_wrong = 0;

void check(const char* what, int a, int b, bool ok) {
    std::printf("%s %d %d %s\n", what, a, b, ok ? "ok" : "WRONG");
    std::fflush(stdout);
    g_wrong += !ok;
}
}  // namespace

extern "C" {
hipError_t hipLaunchCooperativeKernel(const void* f, dim3 g, dim3 b, void** a, unsigned lds, hipStream_t st) {
    static const auto real = (hipError_t(*)(const void*, dim3, dim3, void**, unsigned, hipStream_t))dlsym(
        RTLD_NEXT, "hipLaunchCooperativeKernel");
    g_launches++;
    return real(f, g, b, a, lds, st);
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t lds, hipStream_t st) {
    static const auto real =
        (hipError_t(*)(const void*, dim3, dim3, void**, size_t, hipStream_t))dlsym(RTLD_NEXT, "hipLaunchKernel");
    g_launches++;
    return real(f, g, b, a, lds, st);
}
}

// A hanging cloth of the demo's form with its collider.
struct Cloth {
    oc_verlet v = nullptr;
    int N;
    oc_ellipsoid ball;
    std::vector<float> x, xl, x0;
    Cloth(int nx, int ny) : N(nx * ny), x(3 * N), xl(3 * N), x0(3 * N) {
        unsigned h = 1;
        auto rnd = [&]() { return (float)((h = h * 1664525u + 1013904223u) >> 8) / 16777216.0f - 0.5f; };
        const float d = 4.0f / (float)(std::max(nx, ny) - 1);
        for (int k = 0; k < N; k++) {
            x0[3 * k] = d * (k % nx) - 2.0f + 0.05f * d * rnd();
            x0[3 * k + 1] = 2.0f + 0.05f * d * rnd();
            x0[3 * k + 2] = d * (k / nx) + 0.05f * d * rnd();
        }
        std::vector<oc_spring> sp;
        auto add = [&](int a, int b, float l) { sp.push_back({a, b, l * d, 50.0f, -0.25f, 0}); };
        for (int j = 0; j < ny; j++)
            for (int i = 0; i + 1 < nx; i++) add(j * nx + i, j * nx + i + 1, 1.0f);
        for (int i = 0; i < nx; i++)
            for (int j = 0; j + 1 < ny; j++) add(j * nx + i, (j + 1) * nx + i, 1.0f);
        for (int j = 0; j + 1 < ny; j++)
            for (int i = 0; i + 1 < nx; i++) {
                add(j * nx + i, (j + 1) * nx + i + 1, std::sqrt(2.0f));
                add((j + 1) * nx + i, j * nx + i + 1, std::sqrt(2.0f));
            }
        std::vector<uint8_t> pins(N, 0);
        pins[0] = pins[nx - 1] = 1;
        oc_verlet_params p = {};
        p.mass = 1.0f;
        p.gravity[1] = -0.00981f;
        p.damping = -0.0125f;
        p.dt = 1.0f / 60.0f;
        p.flags = OC_FLAG_GROUND_CLAMP;
        ball = {};
        for (int k = 0; k < 4; k++) ball.transform[5 * k] = ball.inverse[5 * k] = 1.0f;
        ball.center[0] = 0.0f;
        ball.center[1] = 1.9f;
        ball.center[2] = 1.0f;
        ball.radius = 1.0f;
        if (oc_verlet_create(nx, ny, x0.data(), nullptr, sp.data(), (int)sp.size(), pins.data(), &p, &v) != OC_OK)
            std::printf("create: %s\n", oc_last_error());
    }
    ~Cloth() { oc_verlet_destroy(v); }
    bool get() { return oc_verlet_get_state(v, x.data(), xl.data()) == OC_OK; }
    bool same(const Cloth& o) const {
        return std::memcmp(x.data(), o.x.data(), 12 * (size_t)N) == 0 && std::memcmp(xl.data(), o.xl.data(), 12 * (size_t)N) == 0;
    }
};

static void launches() {
    for (int n : {21, 90}) {
        Cloth one(n, n), some(n, n);
        const int steps = 5003;
        g_launches = 0;
        bool ok = oc_verlet_step(one.v, steps, &one.ball) == OC_OK;
        const int many = g_launches;
        for (int left = steps; ok && left > 0; left -= 501)
            ok = oc_verlet_step(some.v, std::min(left, 501), &some.ball) == OC_OK;
        // (at the 6.5 us of the largest cloths, a launch of 2000 steps takes 13 ms)
        check("launches", n, many, ok && many >= steps / 2000 && many < steps / 10 && one.get() && some.get() && one.same(some));
    }
}

static void lost() {
    Cloth c(40, 30), fresh(40, 30);
    int* const err = oc::verlet_error_word(c.v);
    check("error word", 0, 0, err != nullptr);
    if (!err) return;
    auto says = [&](const char* name, int rc) { check(name, rc, OC_ERR_DEVICE, rc == OC_ERR_DEVICE); };
    bool ok = oc_verlet_step(c.v, 8, &c.ball) == OC_OK && c.get();
    *err = 1;
    for (int k = 0; k < 2; k++) {  // not only once
        says("get_state", oc_verlet_get_state(c.v, c.x.data(), c.xl.data()));
        says("get_state of nothing", oc_verlet_get_state(c.v, nullptr, nullptr));
        says("forces", oc_verlet_compute_forces(c.v, c.x.data()));
        says("step", oc_verlet_step(c.v, 8, nullptr));
        says("one step", oc_verlet_step(c.v, 1, nullptr));
        ok = ok && (k ? oc_verlet_set_state(c.v, nullptr, c.x0.data()) : oc_verlet_set_state(c.v, c.x0.data(), nullptr)) == OC_OK;
    }
    // (half a state at a time is none; both arrays are)
    ok = ok && oc_verlet_set_state(c.v, c.x0.data(), c.x0.data()) == OC_OK && oc_verlet_step(c.v, 20, &c.ball) == OC_OK &&
         c.get() && oc_verlet_step(fresh.v, 20, &fresh.ball) == OC_OK && fresh.get();
    check("a new state", 0, 0, ok && c.same(fresh));
}

static void teams() {
    const int sizes[][2] = {{21, 21}, {33, 17}, {130, 100}, {256, 256}, {257, 250}, {512, 512}};
    for (const auto& n : sizes) {
        Cloth one(n[0], n[1]), team(n[0], n[1]);
        const int T = n[0] * n[1] > 256 * 256 || n[0] > 256 ? 32 : 16;
        const int nb = ((n[0] + T - 1) / T) * ((n[1] + T - 1) / T);
        // (0: all of them; teams in turn, so that each set of control words is used after the other)
        for (int blocks : {0, 1, nb / 2, 0, 0, nb - 1, 1}) {
            if (blocks == 0 && nb < 1) continue;
            for (int steps : {2, 5, 4}) {
                const oc_ellipsoid* const e = steps == 4 ? nullptr : &one.ball;
                bool ok = oc::verlet_steps_resident(team.v, steps, e, blocks) == OC_OK;
                for (int k = 0; k < steps; k++) ok = ok && oc_verlet_step(one.v, 1, e) == OC_OK;
                ok = ok && one.get() && team.get();
                check(("team of " + std::to_string(blocks)).c_str(), n[0], n[1], ok && one.same(team));
            }
        }
        check("calls", n[0], n[1], oc_verlet_step(one.v, 12, &one.ball) == OC_OK && oc_verlet_step(team.v, 3, &one.ball) == OC_OK &&
                                       oc_verlet_step(team.v, 9, &one.ball) == OC_OK && one.get() && team.get() && one.same(team));
    }
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "launches") launches();
    else if (what == "lost") lost();
    else if (what == "teams") teams();
    else return 99;
    std::printf("wrong %d\n", g_wrong);
    return g_wrong;
}
