// The tiled PBD plan (pbd_plan.cpp) against the schedule it stands for: one
// solver iteration over the whole cloth, colour by colour, with a mixing
// function in place of the projection (every particle of a constraint takes
// a value that depends on all of them, on the constraint and on its place in
// it).  A block's private copy has to end with the same values at its owned
// particles, and every particle has to be owned once.  Prints one line per
// case: name, accepted, blocks, wrong values.
#include <cstdio>
#include <random>
#include <string>

#include "oc_internal.hpp"

namespace {

using Lists = std::vector<int32_t>;

struct Graph {
    std::vector<float> x;
    Lists d, b;
};

std::vector<int> colour(int N, const Lists& p, int ar, int& ncol) {
    const size_t n = p.size() / ar;
    std::vector<uint64_t> used(N, 0);
    std::vector<int> col(n);
    ncol = 0;
    for (size_t k = 0; k < n; k++) {
        uint64_t m = 0;
        for (int a = 0; a < ar; a++) m |= used[p[ar * k + a]];
        col[k] = __builtin_ctzll(~m);
        for (int a = 0; a < ar; a++) used[p[ar * k + a]] |= uint64_t(1) << col[k];
        ncol = std::max(ncol, col[k] + 1);
    }
    return col;
}

void mix(uint64_t* v, const int32_t* q, int ar, uint64_t tag) {
    uint64_t s = tag, r[3];
    for (int a = 0; a < ar; a++) s = s * 0x9E3779B97F4A7C15ull + v[q[a]];
    for (int a = 0; a < ar; a++) r[a] = (v[q[a]] ^ (s >> (7 + a))) * 0xD1342543DE82EF95ull + s + a;
    for (int a = 0; a < ar; a++) v[q[a]] = r[a];
}

void run(const std::string& name, const Graph& g, int owned, int max_local, float max_work) {
    const int N = (int)g.x.size() / 3;
    oc::PbdFamily f[2];
    std::vector<int> col[2];
    const Lists* lists[2] = {&g.d, &g.b};
    for (int k = 0; k < 2; k++) {
        f[k].arity = 2 + k;
        col[k] = colour(N, *lists[k], 2 + k, f[k].ncol);
        f[k].n = (int)col[k].size();
        f[k].p = lists[k]->data();
        f[k].col = col[k].data();
    }
    oc::PbdPlan P;
    const bool ok = oc::build_pbd_plan(N, g.x.data(), f[0], f[1], owned, max_local, max_work, &P);
    int wrong = 0;
    if (!ok) {
        wrong = P.nb || !P.ids.empty() || !P.rec.empty();
    } else {
        std::vector<uint64_t> whole(N);
        for (int i = 0; i < N; i++) whole[i] = (uint64_t)i * 77 + 5;
        const std::vector<uint64_t> start = whole;
        for (int k = 0; k < 2; k++)
            for (int c = 0; c < f[k].ncol; c++)
                for (int e = 0; e < f[k].n; e++)
                    if (col[k][e] == c) mix(whole.data(), f[k].p + (size_t)f[k].arity * e, f[k].arity, 2 * e + k);
        std::vector<int> owners(N, 0);
        const int ncol = f[0].ncol + f[1].ncol;
        for (int b = 0; b < P.nb; b++) {
            const int nl = P.off[b + 1] - P.off[b];
            if (nl > P.max_local || (P.nb > 1 && nl > max_local) || P.own[b] > nl || P.own[b] > owned) wrong++;
            std::vector<uint64_t> v(nl);
            for (int k = 0; k < nl; k++) v[k] = start[P.ids[P.off[b] + k]];
            for (int c = 0; c < ncol; c++) {
                const int k = c >= f[0].ncol;
                for (int j = P.cptr[(size_t)b * (ncol + 1) + c]; j < P.cptr[(size_t)b * (ncol + 1) + c + 1]; j++) {
                    const int32_t q[3] = {(int32_t)(P.rec[j].ab & 0xFFFF), (int32_t)(P.rec[j].ab >> 16), (int32_t)P.rec[j].c};
                    for (int a = 0; a < f[k].arity; a++)
                        if (q[a] >= nl || P.ids[P.off[b] + q[a]] != f[k].p[(size_t)f[k].arity * P.id[j] + a]) {
                            printf("%s: a record off its constraint\n", name.c_str());
                            return;
                        }
                    mix(v.data(), q, f[k].arity, 2 * (uint64_t)P.id[j] + k);
                }
            }
            for (int k = 0; k < P.own[b]; k++) {
                owners[P.ids[P.off[b] + k]]++;
                if (v[k] != whole[P.ids[P.off[b] + k]]) wrong++;
            }
        }
        for (int n : owners) wrong += n != 1;
    }
    printf("%s %d %d %d\n", name.c_str(), (int)ok, P.nb, wrong);
}

Graph grid(int nx, int ny) {
    Graph g;
    for (int j = 0; j < ny; j++)
        for (int i = 0; i < nx; i++) {
            g.x.insert(g.x.end(), {(float)i, 5.0f, (float)j});
            const int k = j * nx + i;
            if (i + 1 < nx) g.d.insert(g.d.end(), {k, k + 1});
            if (j + 1 < ny) g.d.insert(g.d.end(), {k, k + nx});
            if (i + 1 < nx && j + 1 < ny) g.d.insert(g.d.end(), {k, k + nx + 1, k + nx, k + 1});
            if (i + 2 < nx) g.b.insert(g.b.end(), {k, k + 1, k + 2});
            if (j + 2 < ny) g.b.insert(g.b.end(), {k, k + nx, k + 2 * nx});
        }
    return g;
}

}  // namespace

int main() {
    for (int nx : {1, 2, 3, 21, 64, 130})
        for (int ny : {1, 2, 40, 77})
            for (int owned : {2048, 1024, 100})
                run("grid " + std::to_string(nx) + "x" + std::to_string(ny) + "/" + std::to_string(owned), grid(nx, ny), owned,
                    9216, 1e9f);
    std::mt19937 rng(3);
    for (int t = 0; t < 6; t++) {  // random constraints between near particles, some twice, some of one particle
        Graph g;
        const int N = 700 + 523 * t;
        for (int i = 0; i < 3 * N; i++) g.x.push_back((float)(rng() % 1000));
        for (int k = 0; k < 2 * N; k++) {
            const int a = (int)(rng() % N), b = (a + (int)(rng() % 4)) % N, c = (a + (int)(rng() % 5)) % N;
            g.d.insert(g.d.end(), {a, b});
            if (k % 3 == 0) g.b.insert(g.b.end(), {a, b, c});
        }
        run("near " + std::to_string(N), g, 256, 65536 / 2, 1e9f);
    }
    Graph none = grid(50, 50);
    none.d.clear();
    none.b.clear();
    run("no constraints", none, 1024, 9216, 4.0f);
    Graph points = none;
    std::fill(points.x.begin(), points.x.end(), 1.0f);  // one point: ties everywhere
    run("one point", points, 1024, 9216, 4.0f);
    Graph far = grid(64, 64);  // two families of springs across the cloth
    for (int i = 0; i < 2048; i++) far.d.insert(far.d.end(), {i, 4095 - i, i, i + 2048});
    run("far refused", far, 1024, 3000, 4.0f);
    run("work refused", far, 1024, 9216, 1.0f);
    Graph nan = grid(64, 64);
    nan.x[77] = 0.0f / 0.0f * nan.x[0];
    run("nan refused", nan, 1024, 9216, 4.0f);
    nan.x[77] = 1.0f / 0.0f;
    run("inf refused", nan, 1024, 9216, 4.0f);
    return 0;
}
