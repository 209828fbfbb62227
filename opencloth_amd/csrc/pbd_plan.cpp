// Host-side plan of the tiled PBD solver: particles split into blocks, and
// for each block the constraints it must project, colour by colour, to end
// one solver iteration with the right positions of its own particles.
//
// A solver iteration projects the colours one after another; inside a colour
// no two constraints share a particle.  A block's own particles need the
// last colour's constraints that touch them, these need their other
// particles' values before that colour, and so on back through the colours:
// the block's particle list grows by the constraints' reach per colour (about
// a dozen grid steps on the reference's lists).  Projecting that closure in
// colour order on a private copy gives every owned particle exactly the
// sequence of projections it gets when the colours run over the whole cloth.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <thread>

#include "oc_internal.hpp"

namespace oc {

namespace {

constexpr int kWorkers = 8;

// f() by this thread and up to n - 1 others; false if one ran out of memory.
// A thread that cannot be had is done without.
template <class F>
bool share(int n, const F& f) {
    std::atomic<bool> ok(true);
    auto run = [&]() noexcept {
        try {
            f();
        } catch (...) {
            ok = false;
        }
    };
    std::vector<std::thread> th;
    try {
        for (int t = 1; t < n; t++) th.emplace_back(run);
    } catch (...) {
    }
    run();
    for (auto& t : th) t.join();
    return ok;
}

// Split ids[lo, hi) into nb blocks of nearly equal size: recursive bisection
// along the longer side of the positions' box (ties by id), the block of
// each particle into part.
void bisect(const float* x, int32_t* ids, int lo, int hi, int first, int nb, int* part, int depth) {
    if (nb == 1) {
        for (int k = lo; k < hi; k++) part[ids[k]] = first;
        return;
    }
    float mn[3] = {0, 0, 0}, mx[3] = {0, 0, 0};
    for (int k = lo; k < hi; k++)
        for (int c = 0; c < 3; c++) {
            const float v = x[3 * (size_t)ids[k] + c];
            if (k == lo || v < mn[c]) mn[c] = v;
            if (k == lo || v > mx[c]) mx[c] = v;
        }
    int ax = 0;
    for (int c = 1; c < 3; c++)
        if (mx[c] - mn[c] > mx[ax] - mn[ax]) ax = c;
    const int left = nb / 2;
    const int mid = lo + (int)((int64_t)(hi - lo) * left / nb);
    std::nth_element(ids + lo, ids + mid, ids + hi, [&](int32_t a, int32_t b) {
        const float p = x[3 * (size_t)a + ax], q = x[3 * (size_t)b + ax];
        return p < q || (!(q < p) && a < b);
    });
    std::atomic<int> next(0);
    share(depth > 0 ? 2 : 1, [&]() {
        for (int h; (h = next.fetch_add(1)) < 2;) {
            if (h == 0)
                bisect(x, ids, lo, mid, first, left, part, depth - 1);
            else
                bisect(x, ids, mid, hi, first + left, nb - left, part, depth - 1);
        }
    });
}

bool make_plan(int N, const float* x0, const PbdFamily& dist, const PbdFamily& bend, int owned, int max_local,
               float max_work, PbdPlan& p) {
    for (size_t i = 0; i < 3 * (size_t)N; i++)
        if (!(x0[i] - x0[i] == 0.0f)) return false;  // no order on NaN or infinite positions
    const int nb = std::max(1, (N + owned - 1) / owned);
    const int ncol = dist.ncol + bend.ncol;
    std::vector<int> part(N, 0);
    if (nb > 1) {
        std::vector<int32_t> ids(N);
        for (int i = 0; i < N; i++) ids[i] = i;
        bisect(x0, ids.data(), 0, N, 0, nb, part.data(), 3);
    }
    std::vector<std::vector<int32_t>> own(nb);
    for (int i = 0; i < N; i++) own[part[i]].push_back(i);

    // constraint of colour c at particle q (at most one), -1 if none
    std::vector<int32_t> con((size_t)ncol * N, -1);
    const PbdFamily* fam[2] = {&dist, &bend};
    for (int f = 0; f < 2; f++)
        for (int k = 0; k < fam[f]->n; k++) {
            const int c = fam[f]->col[k] + (f ? dist.ncol : 0);
            for (int a = 0; a < fam[f]->arity; a++)
                con[(size_t)c * N + fam[f]->p[(size_t)fam[f]->arity * k + a]] = k;
        }

    struct Block {
        std::vector<int32_t> ids;                // owned first, then the rest, each by id
        std::vector<std::vector<int32_t>> cons;  // constraints per colour, by id
    };
    std::vector<Block> blk(nb);
    std::atomic<int> next(0);
    std::atomic<bool> ok(true);
    std::atomic<int64_t> work(0);
    auto worker = [&]() {
        std::vector<int> in_list(N, -1);
        std::vector<int> seen[2] = {std::vector<int>(dist.n, -1), std::vector<int>(bend.n, -1)};
        for (int b; ok && (b = next.fetch_add(1)) < nb;) {
            Block& B = blk[b];
            B.ids = own[b];
            B.cons.resize(ncol);
            for (int32_t q : B.ids) in_list[q] = b;
            for (int c = ncol - 1; c >= 0 && ok; c--) {
                const int f = c >= dist.ncol ? 1 : 0, ar = fam[f]->arity;
                const size_t n0 = B.ids.size();
                for (size_t k = 0; k < n0 && ok; k++) {
                    const int32_t e = con[(size_t)c * N + B.ids[k]];
                    if (e < 0 || seen[f][e] == b) continue;
                    seen[f][e] = b;
                    B.cons[c].push_back(e);
                    for (int a = 0; a < ar; a++) {
                        const int32_t q = fam[f]->p[(size_t)ar * e + a];
                        if (in_list[q] != b) {
                            in_list[q] = b;
                            B.ids.push_back(q);
                        }
                    }
                    if ((int)B.ids.size() > max_local) ok = false;  // (for all blocks: the plan is refused)
                }
                work += (int64_t)B.cons[c].size();
            }
            for (int c = 0; c < ncol && ok; c++) {
                const int f = c >= dist.ncol ? 1 : 0, ar = fam[f]->arity;
                std::sort(B.cons[c].begin(), B.cons[c].end(), [&](int32_t x, int32_t y) {
                    const int32_t px = fam[f]->p[(size_t)ar * x], py = fam[f]->p[(size_t)ar * y];
                    return px != py ? px < py : x < y;
                });
            }
            std::sort(B.ids.begin() + own[b].size(), B.ids.end());
        }
    };
    if (!share(std::min(kWorkers, nb), worker) || !ok) return false;
    const int64_t most = INT32_MAX;
    if (work > most || (int64_t)nb * max_local > most || (int64_t)nb * (ncol + 1) > most || (nb > 1 && (double)work > (double)max_work * ((double)dist.n + bend.n)))
        return false;

    p.nb = nb;
    p.off.assign(nb + 1, 0);
    p.own.assign(nb, 0);
    p.cptr.assign((size_t)nb * (ncol + 1), 0);
    int64_t n = 0;
    for (int b = 0; b < nb; b++) {
        p.off[b + 1] = p.off[b] + (int32_t)blk[b].ids.size();
        p.own[b] = (int32_t)own[b].size();
        p.max_local = std::max(p.max_local, (int)blk[b].ids.size());
        for (int c = 0; c <= ncol; c++) {
            p.cptr[(size_t)b * (ncol + 1) + c] = (int32_t)n;
            if (c < ncol) n += (int64_t)blk[b].cons[c].size();
        }
    }
    p.ids.resize(p.off[nb]);
    p.rec.resize(n);
    p.id.resize(n);
    next = 0;
    auto fill = [&]() {
        std::vector<int32_t> local(N, 0);
        for (int b; (b = next.fetch_add(1)) < nb;) {
            const Block& B = blk[b];
            for (size_t k = 0; k < B.ids.size(); k++) {
                local[B.ids[k]] = (int32_t)k;
                p.ids[p.off[b] + k] = B.ids[k];
            }
            size_t o = p.cptr[(size_t)b * (ncol + 1)];
            for (int c = 0; c < ncol; c++) {
                const PbdFamily& f = c < dist.ncol ? dist : bend;
                for (int32_t e : B.cons[c]) {
                    const int32_t* q = f.p + (size_t)f.arity * e;
                    p.rec[o] = {(uint32_t)local[q[0]] | (uint32_t)local[q[1]] << 16, 0.0f,
                                f.arity == 3 ? (uint32_t)local[q[2]] : 0u};
                    p.id[o++] = e;
                }
            }
        }
    };
    return share(std::min(kWorkers, nb), fill);
}

}  // namespace

// Returns false, with an empty plan, when the closures are too large for the
// tiled solver (a block's particles beyond max_local, or more than max_work
// times the constraints of the per-colour form in all), when positions are
// not finite or memory runs out.
bool build_pbd_plan(int N, const float* x0, const PbdFamily& dist, const PbdFamily& bend, int owned, int max_local,
                    float max_work, PbdPlan* out) {
    *out = PbdPlan();
    try {
        if (make_plan(N, x0, dist, bend, owned, max_local, max_work, *out)) return true;
    } catch (...) {
    }
    *out = PbdPlan();
    return false;
}

}  // namespace oc
