// C ABI of the position-based-dynamics cloth (oc_pbd_*): the PBD demo's step
// (OpenCloth_PositionBasedDynamics/.../main.cpp) over caller-given distance
// and bending constraint lists.  Constraints are coloured on the host
// (greedy, in list order: a constraint takes the lowest colour not yet used
// at any of its particles) and laid out for the tiled solver (pbd_plan.cpp):
// one launch per step for a cloth of up to kPbdSmall particles, one per
// solver iteration and two for the sums beyond; constraints that reach too
// far for it are stored colour by colour and one launch projects one colour.
// With OC_FLAG_LIST_ORDER they are stored level by level
// instead (a constraint's level is one more than the highest level among the
// earlier constraints sharing a particle with it) and one single-workgroup
// launch projects all levels of a step in order: the reference's sequential
// results.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "capi_common.hpp"
#include "oc_internal.hpp"

namespace {

using oc::align_up;
using oc::set_error;

float clamp01(float k) { return k > 1.0f ? 1.0f : (k < 0.0f ? 0.0f : k); }

// k' = 1 - (1 - k)^(1/ns), capped at 1 (PBD:153-156, PBD:174-176).
float k_prime(float k, int ns) {
    const float kp = 1.0f - powf(1.0f - k, 1.0f / (float)ns);
    return kp > 1.0f ? 1.0f : kp;
}

// Constraints grouped by group id col[c] (ncol groups): order gets the ids
// group by group, ptr the group offsets.  Inside a group the constraints are
// ordered by first particle: they touch disjoint particles, so the order
// does not change the result, and neighbouring lanes then read neighbouring
// particles (the reference lists column constraints column by column, which
// in list order would put a whole grid row between neighbouring lanes).
void bucket(int N, int n, int arity, const std::vector<int32_t>& p, const std::vector<int>& col, int ncol,
            std::vector<int32_t>& order, std::vector<int32_t>& ptr) {
    ptr.assign((size_t)ncol + 1, 0);
    for (int c = 0; c < n; c++) ptr[col[c] + 1]++;
    for (int k = 0; k < ncol; k++) ptr[k + 1] += ptr[k];
    // by first particle (in list order), then by group, each by counting
    std::vector<int32_t> at((size_t)N + 1, 0), by_first((size_t)n);
    for (int c = 0; c < n; c++) at[p[(size_t)arity * c] + 1]++;
    for (int i = 0; i < N; i++) at[i + 1] += at[i];
    for (int c = 0; c < n; c++) by_first[at[p[(size_t)arity * c]]++] = c;
    std::vector<int32_t> fill(ptr.begin(), ptr.end());
    order.assign((size_t)n, 0);
    for (int32_t c : by_first) order[fill[col[c]]++] = c;
}

// Greedy colouring in list order.  Returns the colour count, -1 past 64.
int colour(int N, int n, int arity, const std::vector<int32_t>& p, std::vector<int>& col) {
    std::vector<uint64_t> used((size_t)N, 0);
    col.assign((size_t)n, 0);
    int ncol = 0;
    for (int c = 0; c < n; c++) {
        uint64_t m = 0;
        for (int a = 0; a < arity; a++) m |= used[p[(size_t)arity * c + a]];
        if (m == ~uint64_t(0)) return -1;
        const int k = __builtin_ctzll(~m);
        col[c] = k;
        for (int a = 0; a < arity; a++) used[p[(size_t)arity * c + a]] |= uint64_t(1) << k;
        ncol = std::max(ncol, k + 1);
    }
    return ncol;
}

// List-order levels: constraint c's level is one more than the highest level
// among the earlier constraints sharing a particle with it, so every earlier
// constraint it depends on sits in a lower level and the constraints of one
// level share no particle.  Returns the level count.
int levels(int N, int n, int arity, const std::vector<int32_t>& p, std::vector<int32_t>& order,
           std::vector<int32_t>& ptr) {
    std::vector<int> last((size_t)N, -1);
    std::vector<int> lev((size_t)n);
    int nlev = 0;
    for (int c = 0; c < n; c++) {
        int l = 0;
        for (int a = 0; a < arity; a++) l = std::max(l, last[p[(size_t)arity * c + a]] + 1);
        lev[c] = l;
        for (int a = 0; a < arity; a++) last[p[(size_t)arity * c + a]] = l;
        nlev = std::max(nlev, l + 1);
    }
    bucket(N, n, arity, p, lev, nlev, order, ptr);
    return nlev;
}

}  // namespace

struct oc_pbd_s {
    int N = 0;
    oc_pbd_params prm{};
    oc::StateIo io;
    hipStream_t stream = nullptr;
    void* arena = nullptr;
    oc::DevPbd dev{};
    std::vector<int32_t> d_ptr, b_ptr;  // colour (or level) offsets, not with the tiled solver
    int n_dcol = 0, n_bcol = 0;         // colours (or levels)
};

namespace {

oc::PbdScalars pscalars(const oc_pbd_s* p) {
    oc::PbdScalars s;
    s.mass = p->prm.mass;
    s.gx = p->prm.gravity[0];
    s.gy = p->prm.gravity[1];
    s.gz = p->prm.gravity[2];
    s.dt = p->prm.dt;
    // InitGL caps global_dampening at 1 and clamps kDamp to [0,1] (PBD:391-396)
    s.gd = p->prm.global_damping > 1.0f ? 1.0f : p->prm.global_damping;
    s.kdamp = clamp01(p->prm.k_damp);
    s.global_k = s.gd * 0.01f;  // PBD:712
    s.inv_dt = 1.0f / p->prm.dt;
    s.flags = p->prm.flags;
    s.w = 1.0f / p->prm.mass;
    const float wsum = s.w + s.w + 2.0f * s.w;
    s.inv_2w = 1.0f / (s.w + s.w);
    s.bend_2w = (2.0f * s.w) / wsum;
    s.bend_4w = (4.0f * s.w) / wsum;
    return s;
}

int check_pbd_params(const oc_pbd_params* p) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "params is NULL");
    if (!(p->mass > 0.0f) || !std::isfinite(p->mass))
        return set_error(OC_ERR_INVALID_ARGUMENT, "mass must be positive");
    if (!(p->dt > 0.0f) || !std::isfinite(p->dt))
        return set_error(OC_ERR_INVALID_ARGUMENT, "dt must be positive");
    if (p->solver_iterations < 1 || p->solver_iterations > 1000)
        return set_error(OC_ERR_INVALID_ARGUMENT, "solver_iterations out of range");
    return OC_OK;
}

}  // namespace

extern "C" {

int oc_pbd_create(int32_t n_vertices, const float* x0, const uint8_t* pinned,
                  const oc_pbd_distance* distance, int32_t n_distance,
                  const oc_pbd_bending* bending, int32_t n_bending, const oc_pbd_params* params,
                  oc_pbd* out) {
    if (!out) return set_error(OC_ERR_INVALID_ARGUMENT, "out is NULL");
    *out = nullptr;
    if (!x0) return set_error(OC_ERR_INVALID_ARGUMENT, "x0 is NULL");
    if (n_vertices < 1 || n_distance < 0 || n_bending < 0)
        return set_error(OC_ERR_INVALID_ARGUMENT, "bad counts");
    if ((n_distance > 0 && !distance) || (n_bending > 0 && !bending))
        return set_error(OC_ERR_INVALID_ARGUMENT, "constraint list is NULL");
    int rc = check_pbd_params(params);
    if (rc != OC_OK) return rc;
    const int N = n_vertices;
    for (int c = 0; c < n_distance; c++) {
        const oc_pbd_distance& d = distance[c];
        if (d.p1 < 0 || d.p1 >= N || d.p2 < 0 || d.p2 >= N || d.p1 == d.p2)
            return set_error(OC_ERR_INVALID_ARGUMENT,
                             "distance constraint " + std::to_string(c) + ": bad particle index");
    }
    for (int c = 0; c < n_bending; c++) {
        const oc_pbd_bending& b = bending[c];
        if (b.p1 < 0 || b.p1 >= N || b.p2 < 0 || b.p2 >= N || b.p3 < 0 || b.p3 >= N ||
            b.p1 == b.p2 || b.p1 == b.p3 || b.p2 == b.p3)
            return set_error(OC_ERR_INVALID_ARGUMENT,
                             "bending constraint " + std::to_string(c) + ": bad particle index");
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return set_error(OC_ERR_NO_DEVICE, "no HIP device");

    // set-up of InitGL (PBD:148-178, PBD:345-351)
    const int ns = params->solver_iterations;
    std::vector<float> W((size_t)N);
    for (int i = 0; i < N; i++) W[i] = (pinned && pinned[i]) ? 0.0f : 1.0f / params->mass;
    std::vector<int32_t> dp(2 * (size_t)n_distance), bp(3 * (size_t)n_bending);
    for (int c = 0; c < n_distance; c++) {
        dp[2 * c] = distance[c].p1;
        dp[2 * c + 1] = distance[c].p2;
    }
    for (int c = 0; c < n_bending; c++) {
        bp[3 * c] = bending[c].p1;
        bp[3 * c + 1] = bending[c].p2;
        bp[3 * c + 2] = bending[c].p3;
    }
    oc_pbd_s* p = new (std::nothrow) oc_pbd_s();
    if (!p) return set_error(OC_ERR_OUT_OF_MEMORY, "host allocation failed");
    std::vector<int32_t> d_order, b_order;
    const bool list_order = (params->flags & OC_FLAG_LIST_ORDER) != 0;
    oc::PbdPlan plan;
    if (list_order) {
        p->n_dcol = levels(N, n_distance, 2, dp, d_order, p->d_ptr);
        p->n_bcol = levels(N, n_bending, 3, bp, b_order, p->b_ptr);
    } else {
        std::vector<int> dcol, bcol;
        p->n_dcol = colour(N, n_distance, 2, dp, dcol);
        p->n_bcol = colour(N, n_bending, 3, bp, bcol);
        if (p->n_dcol < 0 || p->n_bcol < 0) {
            delete p;
            return set_error(OC_ERR_UNSUPPORTED_TOPOLOGY, "constraints need more than 64 colours");
        }
        // the tiled solver where its closures stay small: at most 4 times
        // the constraints (they are 1.7 times on a 512x512 grid of the
        // reference's lists, where a solver iteration takes 10 us against 77
        // us for a launch per colour)
        int dev = 0, lds = 0;
        if (!oc::hip_ok(hipGetDevice(&dev)) ||
            !oc::hip_ok(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)))
            lds = 0;
        const int local = std::min(oc::kPbdLocal, (lds - 4096) / 16);
        const oc::PbdFamily df{n_distance, 2, p->n_dcol, dp.data(), dcol.data()};
        const oc::PbdFamily bf{n_bending, 3, p->n_bcol, bp.data(), bcol.data()};
        const bool small = N <= oc::kPbdSmall;
        if (!oc::build_pbd_plan(N, x0, df, bf, small ? oc::kPbdSmall : oc::kPbdOwned, local, 4.0f, &plan)) {
            bucket(N, n_distance, 2, dp, dcol, p->n_dcol, d_order, p->d_ptr);
            bucket(N, n_bending, 3, bp, bcol, p->n_bcol, b_order, p->b_ptr);
        }
    }
    // rest lengths and k' of every constraint, in list order (PBD:148-178)
    std::vector<float> drest_of((size_t)n_distance), dkp_of((size_t)n_distance), brest_of((size_t)n_bending),
        bkp_of((size_t)n_bending);
    bool d_same = true, b_same = true;  // one k' for the whole family
    auto k_of = [&](float k, size_t c, std::vector<float>& kp, float before, bool& same) {
        kp[c] = c > 0 && k == before ? kp[c - 1] : k_prime(clamp01(k), ns);
        same = same && (c == 0 || std::memcmp(&kp[c], &kp[0], sizeof(float)) == 0);
    };
    for (int c = 0; c < n_distance; c++) {
        const int a = dp[2 * (size_t)c], b = dp[2 * (size_t)c + 1];
        const float dx = x0[3 * a] - x0[3 * b], dy = x0[3 * a + 1] - x0[3 * b + 1],
                    dz = x0[3 * a + 2] - x0[3 * b + 2];
        drest_of[c] = sqrtf(dx * dx + dy * dy + dz * dz);
        k_of(distance[c].k, c, dkp_of, c ? distance[c - 1].k : 0.0f, d_same);
    }
    for (int c = 0; c < n_bending; c++) {
        const int a = bp[3 * (size_t)c], b = bp[3 * (size_t)c + 1], d = bp[3 * (size_t)c + 2];
        float dc[3];
        for (int k = 0; k < 3; k++) {
            const float ctr = 0.3333f * ((x0[3 * a + k] + x0[3 * b + k]) + x0[3 * d + k]);
            dc[k] = x0[3 * d + k] - ctr;
        }
        brest_of[c] = sqrtf(dc[0] * dc[0] + dc[1] * dc[1] + dc[2] * dc[2]);
        k_of(bending[c].k, c, bkp_of, c ? bending[c - 1].k : 0.0f, b_same);
    }

    p->N = N;
    p->prm = *params;
    const int nblk = (N + oc::kPbdBlock - 1) / oc::kPbdBlock;
    oc::DevPbd& d = p->dev;
    d.N = N;
    d.nblk = nblk;
    // device arrays: where each goes, its bytes and its contents (none: zeros)
    struct Array {
        const void** dst;
        size_t bytes;
        const void* src;
    };
    std::vector<Array> arrays;
    auto add = [&](auto*& dst, size_t bytes, const void* src) {
        arrays.push_back({(const void**)(const void*)&dst, std::max<size_t>(bytes, 4), bytes ? src : nullptr});
    };
    const size_t vec = sizeof(float) * 3 * (size_t)N;
    add(d.x, vec, nullptr);
    add(d.v, vec, nullptr);
    add(d.t, vec, nullptr);
    add(d.w, sizeof(float) * (size_t)N, W.data());
    add(d.part, sizeof(float) * oc::kPbdSums * (size_t)nblk, nullptr);
    add(d.sums, sizeof(float) * oc::kPbdSums, nullptr);
    // the constraints in the order they are stored: the plan's records (a
    // constraint once for every block that projects it), or colour by colour
    std::vector<int32_t> d1, d2, b1, b2, b3;
    std::vector<float> drest, dkp, brest, bw, bkp, kp;
    auto bytes_of = [](const auto& v) { return v.size() * sizeof(v[0]); };
    if (plan.nb > 0) {
        d.nb = plan.nb;
        d.nd_col = p->n_dcol;
        d.nb_col = p->n_bcol;
        d.max_local = plan.max_local;
        const int ncol = p->n_dcol + p->n_bcol;
        const bool uniform = d_same && b_same;
        if (!uniform) kp.resize(plan.rec.size());
        for (int b = 0; b < plan.nb; b++)
            for (int c = 0; c < ncol; c++) {
                const int32_t* at = plan.cptr.data() + (size_t)b * (ncol + 1) + c;
                for (int32_t j = at[0]; j < at[1]; j++) {
                    const int32_t e = plan.id[j];
                    plan.rec[j].rest = c < p->n_dcol ? drest_of[e] : brest_of[e];
                    if (!uniform) kp[j] = c < p->n_dcol ? dkp_of[e] : bkp_of[e];
                }
            }
        if (plan.rec.empty()) plan.rec.push_back({0u, 0.0f, 0u});  // (what an idle thread loads)
        d.n_rec = (int)plan.rec.size();
        add(d.t_off, bytes_of(plan.off), plan.off.data());
        add(d.t_own, bytes_of(plan.own), plan.own.data());
        add(d.t_ids, bytes_of(plan.ids), plan.ids.data());
        add(d.t_cptr, bytes_of(plan.cptr), plan.cptr.data());
        add(d.t_rec, bytes_of(plan.rec), plan.rec.data());
        if (!uniform) add(d.t_kp, bytes_of(kp), kp.data());
        d.d_kp_all = n_distance > 0 ? dkp_of[0] : 0.0f;
        d.b_kp_all = n_bending > 0 ? bkp_of[0] : 0.0f;
        if (plan.nb > 1) add(d.t2, vec, nullptr);
    } else {
        for (int32_t c : d_order) {
            drest.push_back(drest_of[c]);
            dkp.push_back(dkp_of[c]);
            d1.push_back(dp[2 * (size_t)c]);
            d2.push_back(dp[2 * (size_t)c + 1]);
        }
        for (int32_t c : b_order) {
            brest.push_back(brest_of[c]);
            bkp.push_back(bkp_of[c]);
            const int a = bp[3 * (size_t)c], b = bp[3 * (size_t)c + 1], e = bp[3 * (size_t)c + 2];
            b1.push_back(a);
            b2.push_back(b);
            b3.push_back(e);
            bw.push_back(W[a] + W[b] + 2.0f * W[e]);
        }
        add(d.d_p1, bytes_of(d1), d1.data());
        add(d.d_p2, bytes_of(d2), d2.data());
        add(d.d_rest, bytes_of(drest), drest.data());
        add(d.d_kp, bytes_of(dkp), dkp.data());
        add(d.b_p1, bytes_of(b1), b1.data());
        add(d.b_p2, bytes_of(b2), b2.data());
        add(d.b_p3, bytes_of(b3), b3.data());
        add(d.b_rest, bytes_of(brest), brest.data());
        add(d.b_w, bytes_of(bw), bw.data());
        add(d.b_kp, bytes_of(bkp), bkp.data());
        add(d.d_lv, bytes_of(p->d_ptr), p->d_ptr.data());
        add(d.b_lv, bytes_of(p->b_ptr), p->b_ptr.data());
        d.nd_lv = (int)p->d_ptr.size() - 1;
        d.nb_lv = (int)p->b_ptr.size() - 1;
    }
    size_t total = 0;
    for (const Array& a : arrays) total += align_up(a.bytes);
    if (hipMalloc(&p->arena, total) != hipSuccess) {
        delete p;
        return set_error(OC_ERR_OUT_OF_MEMORY, "hipMalloc failed");
    }
    bool ok = hipMemset(p->arena, 0, total) == hipSuccess;
    char* q = (char*)p->arena;
    for (const Array& a : arrays) {
        *a.dst = q;
        if (ok && a.src) ok = hipMemcpy(q, a.src, a.bytes, hipMemcpyHostToDevice) == hipSuccess;
        q += align_up(a.bytes);
    }
    if (!ok) {
        (void)hipFree(p->arena);
        delete p;
        return set_error(OC_ERR_DEVICE, "upload failed");
    }
    p->io.prepare((size_t)N, 3);
    *out = p;
    rc = oc_pbd_set_state(p, x0, nullptr);
    if (rc != OC_OK) {
        std::string e = oc_last_error();
        oc_pbd_destroy(p);
        *out = nullptr;
        return set_error(rc, e);
    }
    return OC_OK;
}

int oc_pbd_destroy(oc_pbd p) {
    if (!p) return OC_OK;
    (void)hipStreamSynchronize(p->stream);
    if (p->arena) (void)hipFree(p->arena);
    delete p;
    return OC_OK;
}

int oc_pbd_set_stream(oc_pbd p, void* stream) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "pbd is NULL");
    p->stream = (hipStream_t)stream;
    return OC_OK;
}

// x and v may be NULL to keep that vector, except that v defaults to zero on
// the first call from oc_pbd_create.
int oc_pbd_set_state(oc_pbd p, const float* x, const float* v) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "pbd is NULL");
    const size_t N = (size_t)p->N;
    OC_HIP(p->io.write({{x ? p->dev.x : nullptr, N, const_cast<float*>(x)},
                        {v ? p->dev.v : nullptr, N, const_cast<float*>(v)}}, p->stream));
    return OC_OK;
}

int oc_pbd_get_state(oc_pbd p, float* x, float* v) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "pbd is NULL");
    const size_t N = (size_t)p->N;
    OC_HIP(p->io.read({{p->dev.x, N, x}, {p->dev.v, N, v}}, p->stream));
    return OC_OK;
}

int oc_pbd_num_colors(oc_pbd p, int32_t* n_distance_colors, int32_t* n_bending_colors) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "pbd is NULL");
    if (n_distance_colors) *n_distance_colors = p->n_dcol;
    if (n_bending_colors) *n_bending_colors = p->n_bcol;
    return OC_OK;
}

int oc_pbd_step(oc_pbd p, int32_t nsteps, const oc_ellipsoid* e) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "pbd is NULL");
    if (nsteps < 0) return set_error(OC_ERR_INVALID_ARGUMENT, "nsteps < 0");
    const oc::PbdScalars s = pscalars(p);
    const oc::DevPbd& d = p->dev;
    if (d.nb == 1) {
        const int most = 1024 / p->prm.solver_iterations + 1;  // steps of one launch: up to some 10 ms
        for (int left = nsteps; left > 0; left -= most)
            OC_HIP(oc::launch_pbd_small(d, s, std::min(most, left), p->prm.solver_iterations, e, p->stream));
        return OC_OK;
    }
    if (d.nb > 1) {
        for (int n = 0; n < nsteps; n++) OC_HIP(oc::launch_pbd_tiled(d, s, p->prm.solver_iterations, e, p->stream));
        return OC_OK;
    }
    const int nd_col = p->n_dcol, nb_col = p->n_bcol;
    for (int n = 0; n < nsteps; n++) {
        if (p->prm.flags & OC_FLAG_LIST_ORDER) {
            OC_HIP(oc::launch_pbd_predict_seq(d, s, p->stream));
            OC_HIP(oc::launch_pbd_levels(d, s, p->prm.solver_iterations,
                                         (p->prm.flags & OC_FLAG_GROUND_CLAMP) ? 1 : 0, p->stream));
        } else {
            OC_HIP(oc::launch_pbd_predict(d, s, p->stream));
            for (int it = 0; it < p->prm.solver_iterations; it++) {
                for (int c = 0; c < nd_col; c++)
                    OC_HIP(oc::launch_pbd_distance(d, s, p->d_ptr[c], p->d_ptr[c + 1] - p->d_ptr[c], p->stream));
                for (int c = 0; c < nb_col; c++)
                    OC_HIP(oc::launch_pbd_bending(d, s, p->b_ptr[c], p->b_ptr[c + 1] - p->b_ptr[c], p->stream));
                if (p->prm.flags & OC_FLAG_GROUND_CLAMP) OC_HIP(oc::launch_pbd_ground(d, p->stream));
            }
        }
        if (e) OC_HIP(oc::launch_ellipsoid(d.t, d.v, d.N, *e, 0, p->stream));
        OC_HIP(oc::launch_pbd_integrate(d, s, p->stream));
    }
    return OC_OK;
}

int oc_pbd_synchronize(oc_pbd p) {
    if (!p) return set_error(OC_ERR_INVALID_ARGUMENT, "pbd is NULL");
    OC_HIP(hipStreamSynchronize(p->stream));
    return OC_OK;
}

}  // extern "C"
