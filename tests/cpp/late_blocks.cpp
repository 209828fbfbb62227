// Blocks of the resident solve that start after its roll was closed: one
// block starts a solve alone, and a few milliseconds later others come on
// another stream (too few in all for the roll to fill).  Prints the solve's
// time with the one block and with the late ones, and whether iterations,
// status and solution are those of a complete team.  argv: nx ny max_iters
// tol_mode.
#define main resident_team_main
#include "resident_team.cpp"
#undef main

#include <chrono>
#include <thread>

int main(int argc, char** argv) {
    if (argc != 5) return 2;
    const int nx = std::atoi(argv[1]), ny = std::atoi(argv[2]), its = std::atoi(argv[3]), mode = std::atoi(argv[4]);
    const int N = nx * ny;
    std::vector<float> X(3 * N), V(3 * N);
    unsigned h = 1;
    auto rnd = [&]() { return (float)((h = h * 1664525u + 1013904223u) >> 8) / 16777216.0f - 0.5f; };
    for (int k = 0; k < N; k++) {
        X[3 * k] = 0.01f * (k % nx);
        X[3 * k + 1] = 0.0f;
        X[3 * k + 2] = 0.01f * (k / nx);
    }
    const std::vector<oc_spring> sp = grid_springs(nx, ny, X);
    for (float& x : X) x += 1e-4f * rnd();
    for (float& v : V) v = 0.1f * rnd();
    oc_params p = {};
    p.mass = 1.0f;
    p.gravity[1] = -9.81f;
    p.dt = 1.0f / 60.0f;
    p.cg_max_iters = its;
    p.cg_tol = 1e-4f;
    p.cg_tol_mode = mode;
    oc_cloth c = nullptr;
    if (oc_cloth_create(nx, ny, X.data(), V.data(), sp.data(), (int)sp.size(), nullptr, &p, &c) != OC_OK) return 1;
    const oc::DevCloth& d = oc::cloth_view(c);
    const int nb = oc::resident_blocks(d.ntx, d.nty, d.res_vt);
    oc::StepScalars s{};
    s.mass = s.md = p.mass;
    s.gy = p.gravity[1];
    s.h = p.dt;
    s.hh = p.dt * p.dt;
    s.tol2 = p.cg_tol * p.cg_tol;
    s.max_it = its;
    s.tol_mode = mode;
    hipStream_t one, two;
    if (!d.res_vt || hipStreamCreateWithFlags(&one, hipStreamNonBlocking) != hipSuccess ||
        hipStreamCreateWithFlags(&two, hipStreamNonBlocking) != hipSuccess)
        return 1;
    std::vector<float> dv[3];
    int it[3] = {}, st[3] = {};
    double us[3] = {};
    const int late = nb - 2;  // with the first block still one too few
    for (int k = 0; k < 3; k++) {  // a complete team, one block, one block and late ones
        dv[k].resize(3 * N);
        if (oc_cloth_set_dv(c, nullptr) != OC_OK || oc_cloth_assemble(c, p.dt) != OC_OK ||
            hipDeviceSynchronize() != hipSuccess)
            return 1;
        const auto t0 = std::chrono::steady_clock::now();
        if (oc::launch_cg_resident(d, s, one, true, k == 0 ? nb : 1) != hipSuccess) return 1;
        if (k == 2) {
            std::this_thread::sleep_for(std::chrono::milliseconds(4));
            if (oc::launch_cg_resident(d, s, two, true, late) != hipSuccess) return 1;
        }
        if (hipDeviceSynchronize() != hipSuccess) return 1;
        us[k] = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
        if (oc_cloth_last_status(c, &it[k], &st[k]) != OC_OK || oc_cloth_get_dv(c, dv[k].data()) != OC_OK) return 1;
    }
    for (int k = 1; k < 3; k++)
        std::printf("%s: %d %d %d %d same %d us %.0f\n", k == 1 ? "one block" : "late blocks", it[0], st[0], it[k], st[k],
                    std::memcmp(dv[0].data(), dv[k].data(), 12 * (size_t)N) == 0, us[k]);
    (void)hipStreamDestroy(one);
    (void)hipStreamDestroy(two);
    return oc_cloth_destroy(c) == OC_OK ? 0 : 1;
}
