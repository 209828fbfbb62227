// The resident solve's partial team: the same assembled system solved with
// every block, and with fewer blocks than regions, so that the roll call
// never completes, is closed after its time limit, and the blocks that
// signed in run the solve with the memory-based phases.  Prints one line per
// team size: iterations and status of both solves, and whether the solutions
// are the same bits.  argv: nx ny max_iters tol_mode.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "oc_internal.hpp"

static std::vector<oc_spring> grid_springs(int nx, int ny, const std::vector<float>& X) {
    std::vector<oc_spring> sp;
    auto add = [&](int a, int b) {
        float d2 = 0.0f;
        for (int c = 0; c < 3; c++) {
            const float d = X[3 * a + c] - X[3 * b + c];
            d2 += d * d;
        }
        sp.push_back({a, b, std::sqrt(d2), 50.0f, -0.25f, 0});
    };
    for (int j = 0; j < ny; j++)
        for (int i = 0; i + 1 < nx; i++) add(j * nx + i, j * nx + i + 1);
    for (int i = 0; i < nx; i++)
        for (int j = 0; j + 1 < ny; j++) add(j * nx + i, (j + 1) * nx + i);
    for (int j = 0; j + 1 < ny; j++)
        for (int i = 0; i + 1 < nx; i++) {
            add(j * nx + i, (j + 1) * nx + i + 1);
            add((j + 1) * nx + i, j * nx + i + 1);
        }
    for (int j = 0; j < ny; j++)
        for (int i = 0; i + 2 < nx; i++) add(j * nx + i, j * nx + i + 2);
    for (int i = 0; i < nx; i++)
        for (int j = 0; j + 2 < ny; j++) add(j * nx + i, (j + 2) * nx + i);
    return sp;
}

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
    std::vector<uint8_t> pins(N, 0);
    for (int i = 0; i < nx; i++) pins[i] = 1;
    oc_params p = {};
    p.mass = 1.0f;
    p.gravity[1] = -9.81f;
    p.dt = 1.0f / 60.0f;
    p.cg_max_iters = its;
    p.cg_tol = 1e-4f;
    p.cg_tol_mode = mode;
    oc_cloth c = nullptr;
    if (oc_cloth_create(nx, ny, X.data(), V.data(), sp.data(), (int)sp.size(), pins.data(), &p, &c) != OC_OK) {
        std::printf("create: %s\n", oc_last_error());
        return 1;
    }
    const oc::DevCloth& d = oc::cloth_view(c);
    if (!d.res_vt) {
        std::printf("no resident solve for this cloth\n");
        return 1;
    }
    const int nb = oc::resident_blocks(d.ntx, d.nty, d.res_vt);
    oc::StepScalars s{};
    s.mass = s.md = p.mass;
    s.gy = p.gravity[1];
    s.h = p.dt;
    s.hh = p.dt * p.dt;
    s.tol2 = p.cg_tol * p.cg_tol;
    s.max_it = its;
    s.tol_mode = mode;
    std::vector<float> full(3 * N), part(3 * N);
    const int teams[] = {nb, 1, nb / 2, nb - 1};
    int it0 = 0, st0 = 0;
    for (int blocks : teams) {
        if (blocks < 1) continue;
        int it = 0, st = 0;
        if (oc_cloth_set_dv(c, nullptr) != OC_OK || oc_cloth_assemble(c, p.dt) != OC_OK ||
            oc::launch_cg_resident(d, s, nullptr, true, blocks) != hipSuccess ||
            oc_cloth_last_status(c, &it, &st) != OC_OK ||
            oc_cloth_get_dv(c, blocks == nb ? full.data() : part.data()) != OC_OK) {
            std::printf("team %d: %s\n", blocks, oc_last_error());
            return 1;
        }
        if (blocks == nb) {
            it0 = it;
            st0 = st;
            part = full;
        }
        std::printf("team %d of %d: %d %d %d %d same %d\n", blocks, nb, it0, st0, it, st,
                    std::memcmp(full.data(), part.data(), 12 * (size_t)N) == 0);
        std::fflush(stdout);
    }
    return oc_cloth_destroy(c) == OC_OK ? 0 : 1;
}
