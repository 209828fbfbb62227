// Device-side helpers shared by the single-cloth and batched kernels:
// vec3 arithmetic in the reference's GLM expression order, the per-spring
// force/Jacobian, and the fixed-order reductions.  Built with
// -ffp-contract=off, so every expression rounds exactly as written.
#pragma once

#include "oc_internal.hpp"

namespace oc {
namespace dev {

constexpr int kPartialRegs = 16;  // tile partials per lane loaded up front

// Blocks are dispatched round-robin over the 8 XCDs; each XCD gets a
// contiguous band of tiles so that halo and shared-data re-reads hit its L2.
__device__ inline int tile_of_block(int b, int nt) {
    if ((nt & 7) == 0) return (b & 7) * (nt >> 3) + (b >> 3);
    return b;
}

struct V3 {
    float x, y, z;
};

__device__ inline V3 ld3(const float* p, int N, int i) { return {p[i], p[N + i], p[2 * N + i]}; }
__device__ inline void st3(float* p, int N, int i, V3 v) {
    p[i] = v.x;
    p[N + i] = v.y;
    p[2 * N + i] = v.z;
}

// Element idx of a device array, addressed by a 32-bit byte offset from the
// array's base.  With a uniform base this is the scalar-base form of a global
// load (no 64-bit address arithmetic per element).  Callers guarantee that
// the array is below 4 GiB (checked when a cloth is created).
template <typename T>
__device__ inline T ldo(const T* p, uint32_t idx) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + idx * (uint32_t)sizeof(T));
}
template <typename T>
__device__ inline void sto(T* p, uint32_t idx, T v) {
    *reinterpret_cast<T*>(reinterpret_cast<char*>(p) + idx * (uint32_t)sizeof(T)) = v;
}
// SoA vec3 with the component planes as uniform bases: one 32-bit offset
// serves all three components.
__device__ inline V3 ld3o(const float* p, int N, int i) {
    return {ldo(p, (uint32_t)i), ldo(p + N, (uint32_t)i), ldo(p + 2 * (size_t)N, (uint32_t)i)};
}
__device__ inline void st3o(float* p, int N, int i, V3 v) {
    sto(p, (uint32_t)i, v.x);
    sto(p + N, (uint32_t)i, v.y);
    sto(p + 2 * (size_t)N, (uint32_t)i, v.z);
}
__device__ inline V3 add3(V3 a, V3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ inline V3 sub3(V3 a, V3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ inline V3 scl3(float s, V3 a) { return {s * a.x, s * a.y, s * a.z}; }
__device__ inline float dot3(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
// symmetric (xx,yy,zz,xy,xz,yz) times vector, mat3*vec3 order
__device__ inline V3 symmv(const float* c, V3 w) {
    return {c[0] * w.x + c[3] * w.y + c[4] * w.z, c[3] * w.x + c[1] * w.y + c[5] * w.z,
            c[4] * w.x + c[5] * w.y + c[2] * w.z};
}

// Force on p1 (OpenCloth_ImplicitEuler/.../main.cpp:663-675), stiffness
// Jacobian K (:669-671) and P = dp dp^T / l^2, in the reference's expression
// order.
__device__ inline void spring_terms(V3 x1, V3 x2, V3 v1, V3 v2, float L0, float Ks, float Kd,
                                    V3& f, float* K, float* P) {
    V3 dp = {x1.x - x2.x, x1.y - x2.y, x1.z - x2.z};
    V3 dv = {v1.x - v2.x, v1.y - v2.y, v1.z - v2.z};
    float sq = dp.x * dp.x + dp.y * dp.y + dp.z * dp.z;
    float dist = sqrtf(sq);
    float dist2 = dist * dist;
    float lo_l = L0 / dist;
    P[0] = (dp.x * dp.x) / dist2;
    P[1] = (dp.y * dp.y) / dist2;
    P[2] = (dp.z * dp.z) / dist2;
    P[3] = (dp.y * dp.x) / dist2;
    P[4] = (dp.z * dp.x) / dist2;
    P[5] = (dp.z * dp.y) / dist2;
#pragma unroll
    for (int c = 0; c < 3; c++) K[c] = Ks * (-1.0f + lo_l * (1.0f - P[c]));
#pragma unroll
    for (int c = 3; c < 6; c++) K[c] = Ks * (lo_l * (0.0f - P[c]));
    float leftTerm = -Ks * (dist - L0);
    float rightTerm = Kd * ((dv.x * dp.x + dv.y * dp.y + dv.z * dp.z) / dist);
    float inv = 1.0f / sqrtf(sq);
    float s = leftTerm + rightTerm;
    f = {s * (dp.x * inv), s * (dp.y * inv), s * (dp.z * inv)};
}

// One spring from the x1 end: force on x1, K (v1 - v2) and the pair-block
// term h (kd P) + h^2 K, in the per-end assembly's expressions.
struct SpringOut {
    V3 f, kw;
    float c[6];
};
__device__ inline SpringOut eval_spring(V3 x1, V3 x2, V3 v1, V3 v2, float L0, float ks, float kd,
                                        float h, float hh) {
    SpringOut o;
    float K[6], P[6];
    spring_terms(x1, x2, v1, v2, L0, ks, kd, o.f, K, P);
#pragma unroll
    for (int q = 0; q < 6; q++) o.c[q] = h * (kd * P[q]) + hh * K[q];
    o.kw = symmv(K, V3{v1.x - v2.x, v1.y - v2.y, v1.z - v2.z});
    return o;
}

// Force only (no Jacobian), same arithmetic as spring_terms.
__device__ inline V3 spring_force(V3 x1, V3 x2, V3 v1, V3 v2, float L0, float Ks, float Kd) {
    V3 dp = {x1.x - x2.x, x1.y - x2.y, x1.z - x2.z};
    V3 dv = {v1.x - v2.x, v1.y - v2.y, v1.z - v2.z};
    float sq = dp.x * dp.x + dp.y * dp.y + dp.z * dp.z;
    float dist = sqrtf(sq);
    float leftTerm = -Ks * (dist - L0);
    float rightTerm = Kd * ((dv.x * dp.x + dv.y * dp.y + dv.z * dp.z) / dist);
    float inv = 1.0f / sqrtf(sq);
    float s = leftTerm + rightTerm;
    return {s * (dp.x * inv), s * (dp.y * inv), s * (dp.z * inv)};
}

// v, opaque to the compiler: what is computed from it is not moved ahead of
// an iteration loop, where a few dozen addresses would spill.
__device__ inline unsigned here(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Word i of an exchange between blocks, from a uniform base and a 32-bit offset.
__device__ inline uint64_t xch_load(const uint64_t* p, unsigned i) {
    return __hip_atomic_load(reinterpret_cast<const uint64_t*>(reinterpret_cast<const char*>(p) + here(i * 8u)),
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xch_store(uint64_t* p, unsigned i, unsigned tag, float v) {
    __hip_atomic_store(reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(p) + here(i * 8u)),
                       ((uint64_t)tag << 32) | (uint64_t)__float_as_uint(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Roll call of a launch whose blocks wait for each other, and so must all run.
constexpr unsigned kRollClosed = 1u << 15;       // the count is in bits 0-14
// How long blocks wait for the others: about what an incomplete team takes
// longer than a complete one (512x512, 30 iterations: 0.24 ms complete, 1.75
// by tickets with half of the blocks or all but one; 128x128, 40 iterations:
// 0.17 and 0.7).  Beside another stream's products that leave CUs only now and
// then, a 512x512 step takes 0.82 ms; with half the wait, and without the late
// blocks, it took 1.95.
constexpr unsigned long long kRollCallTicks = 100000;  // 1 ms of the 100 MHz counter
// Sign in (one thread per block), then wait until all nb blocks have: true
// once they have, false when the roll is closed.  The word decides: a close
// only succeeds on a word whose count is below nb, and once the count has
// reached nb no block closes it.
__device__ inline void roll_call_sign(unsigned* roll) {
    __hip_atomic_fetch_add(roll, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool roll_call_wait(unsigned* roll, int nb) {
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
        unsigned w = __hip_atomic_load(roll, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (w & kRollClosed) return false;
        if ((int)w >= nb) return true;
        if (__builtin_amdgcn_s_memrealtime() - t0 > kRollCallTicks)
            __hip_atomic_compare_exchange_strong(roll, &w, w | kRollClosed, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        else
            __builtin_amdgcn_s_sleep(1);
    }
}

// Phases of `pieces` pieces of work each, for blocks that need not all be
// running: a block takes the next ticket (phase by phase), waits until the
// phases before its own are complete, does the piece and says so.  A ticket's
// holder only waits for holders of earlier tickets, which are running, so any
// number of blocks gets through, a single one too, and blocks that start late
// take part from then on.  q[0]: tickets taken, q[kTicketDone]: pieces done (a
// cache line of its own), both zero at the start.  *stop, set while a piece is done, ends the work in the next
// phase at the latest.  A wait is bounded; on time-out *err is set and the
// block leaves, so every wave exits.  A launch has fewer than 2^31 pieces.
enum { kTicketWork, kTicketLast, kTicketOver };
struct Ticket {
    unsigned n;
    int what;
};
constexpr unsigned kTicketPolls = 1u << 22;  // seconds
// The block's next ticket t: a piece of work (t.n counts over all phases);
// the one after the last piece, which a single block gets, once all are done;
// or nothing more to do.  What other blocks wrote in earlier phases is visible.
__device__ inline int ticket_take(unsigned* q, unsigned pieces, unsigned total, int* stop, int* err, Ticket& t) {
    __syncthreads();  // t and the last piece's shared memory are free
    if (threadIdx.x == 0) {
        const unsigned n = __hip_atomic_fetch_add(q, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int what = n < total ? kTicketWork : n == total ? kTicketLast : kTicketOver;
        auto stopped = [&]() { return stop && __hip_atomic_load(stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
        if (what != kTicketOver) {
            unsigned polls = 0;
            while (__hip_atomic_load(q + kTicketDone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n / pieces * pieces) {
                if (stopped()) break;
                if (++polls > kTicketPolls) {
                    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    what = kTicketOver;
                    break;
                }
                __builtin_amdgcn_s_sleep(8);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            if (stopped()) what = kTicketOver;
        }
        t.n = n;
        t.what = what;
    }
    __syncthreads();
    return t.what;
}
// The block's piece is done: its writes first (every wave's, then the release
// takes them to the device-coherent level).
__device__ inline void ticket_done(unsigned* q) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_fetch_add(q + kTicketDone, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

// Wave tree: lane l += lane l+off for off = 32..1; lane 0 ends with the sum
// (the other lanes' values are not the tree's).  Offsets 32 and 16 by gfx950's
// lane-swap instructions, the rest by row shifts inside 16 lanes: register
// moves of a few cycles, where each __shfl_down is an LDS round trip.
template <int N>
__device__ inline float row_down(float t) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(t), 0x100 + N, 0xF, 0xF, true));
}
__device__ inline float wave_sum(float t) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    t += __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(t), __float_as_uint(t), false, false);
    t += __uint_as_float(b[1]);
    t += row_down<8>(t);
    t += row_down<4>(t);
    t += row_down<2>(t);
    t += row_down<1>(t);
    return t;
}

// Tile partial: wave sums added in wave order.  Result valid in thread 0.
template <int NT>
__device__ inline float tile_sum(float t, float* ws) {
    t = wave_sum(t);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) ws[w] = t;
    __syncthreads();
    float p = 0.0f;
    if (threadIdx.x == 0) {
        p = ws[0];
#pragma unroll
        for (int k = 1; k < NT / 64; k++) p = p + ws[k];
    }
    return p;
}

// Cross-tile sum in two halves so the loads can be issued early.  Lane l of
// wave 0 sums tiles l, l+64, l+128, ... in order, then the wave tree.
__device__ inline void partial_load(const float* part, int nt, float* v) {
#pragma unroll
    for (int j = 0; j < kPartialRegs; j++) {
        const int k = threadIdx.x + 64 * j;
        v[j] = k < nt ? part[k] : 0.0f;
    }
}
__device__ inline float partial_finish(const float* part, int nt, const float* v) {
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < kPartialRegs; j++) s += v[j];
    for (int k = threadIdx.x + 64 * kPartialRegs; k < nt; k += 64) s += part[k];
    return wave_sum(s);
}

// Sum of nt tile partials, returned to all threads (one-shot form).
__device__ inline float partial_sum(const float* part, int nt, float* bc) {
    if (threadIdx.x < 64) {
        float v[kPartialRegs];
        partial_load(part, nt, v);
        const float s = partial_finish(part, nt, v);
        if (threadIdx.x == 0) *bc = s;
    }
    __syncthreads();
    return *bc;
}

// EllipsoidCollision (OpenCloth_ImplicitEuler/.../main.cpp:727-751) of one
// point: its place on the surface when p is inside, p otherwise.
__device__ __forceinline__ V3 ellipsoid_push(const oc_ellipsoid& e, V3 p, bool& inside) {
    float d0[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const float t = e.inverse[0 * 4 + r] * p.x + e.inverse[1 * 4 + r] * p.y +
                        e.inverse[2 * 4 + r] * p.z + e.inverse[3 * 4 + r] * 1.0f;
        d0[r] = t - e.center[r];
    }
    const float dist = sqrtf(d0[0] * d0[0] + d0[1] * d0[1] + d0[2] * d0[2]);
    inside = dist < 1.0f;
    if (!inside) return p;
#pragma unroll
    for (int c = 0; c < 3; c++) d0[c] = ((e.radius - dist) * d0[c]) / dist;
    float delta[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        float t[3] = {e.transform[0 * 4 + a], e.transform[1 * 4 + a], e.transform[2 * 4 + a]};
        const float tt = t[0] * t[0] + t[1] * t[1] + t[2] * t[2];
#pragma unroll
        for (int c = 0; c < 3; c++) t[c] = t[c] / tt;
        delta[a] = d0[0] * t[0] + d0[1] * t[1] + d0[2] * t[2];
    }
    return {p.x + delta[0], p.y + delta[1], p.z + delta[2]};
}

// Per-spring adjoint terms (oracle.c spring_adjoint, same expression order):
// derivative of h mu.f + h^2 mu.K v' + h mu.D dv with respect to e = x1-x2
// (ge), to v1 (gvv) and to ks (gk).
__device__ inline void spring_adjoint(V3 xa, V3 xb, V3 va, V3 vb, V3 ua, V3 ub, V3 wa, V3 wb,
                                      V3 pa, V3 pb, float L0, float ks, float Kd, float h, float hh,
                                      float* ge, float* gvv, float& gk) {
    const float e[3] = {xa.x - xb.x, xa.y - xb.y, xa.z - xb.z};
    const float dvel[3] = {va.x - vb.x, va.y - vb.y, va.z - vb.z};
    const float u[3] = {ua.x - ub.x, ua.y - ub.y, ua.z - ub.z};
    const float w[3] = {wa.x - wb.x, wa.y - wb.y, wa.z - wb.z};
    const float wp[3] = {pa.x - pb.x, pa.y - pb.y, pa.z - pb.z};
    const float l = sqrtf(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
    const float il = 1.0f / l;
    const float il2 = il * il, il3 = il2 * il, il4 = il2 * il2, il5 = il4 * il;
    const float ue = u[0] * e[0] + u[1] * e[1] + u[2] * e[2];
    const float we = w[0] * e[0] + w[1] * e[1] + w[2] * e[2];
    const float wpe = wp[0] * e[0] + wp[1] * e[1] + wp[2] * e[2];
    const float uw = u[0] * w[0] + u[1] * w[1] + u[2] * w[2];
    const float dve = dvel[0] * e[0] + dvel[1] * e[1] + dvel[2] * e[2];
    const float phi = -ks * (l - L0) + Kd * (dve * il);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const float dphi = -ks * e[c] * il + Kd * (dvel[c] * il - dve * e[c] * il3);
        const float A = h * ((ue * il) * dphi + phi * (u[c] * il - ue * e[c] * il3));
        const float B = hh * ks * L0 *
                        (-uw * e[c] * il3 - (u[c] * we + w[c] * ue) * il3 + 3.0f * ue * we * e[c] * il5);
        const float Cc = h * Kd * ((u[c] * wpe + wp[c] * ue) * il2 - 2.0f * ue * wpe * e[c] * il4);
        ge[c] = A + B + Cc;
    }
    V3 f;
    float K[6], P[6];
    spring_terms(xa, xb, va, vb, L0, ks, Kd, f, K, P);
    const V3 ku = symmv(K, V3{u[0], u[1], u[2]});
    gvv[0] = h * Kd * ue * e[0] * il2 + hh * ku.x;
    gvv[1] = h * Kd * ue * e[1] * il2 + hh * ku.y;
    gvv[2] = h * Kd * ue * e[2] * il2 + hh * ku.z;
    gk = h * (ue * il) * (-(l - L0)) + hh * ((L0 * il - 1.0f) * uw - L0 * ue * we * il3);
}

// What the adjoint gather reads: pre-step x, v, the adjoint solve mu and the
// step's solution p (planes of stride N), the assembly slots (slot-major).
struct AdjGatherIn {
    const float* x;
    const float* v;
    const float* mu;
    const float* p;
    const int32_t* ainc_s;
    const uint16_t* ainc_m;
    int N, wa;
};

// Adjoint gather of vertex i: the spring terms of dJ/dx into gx, of dJ/dv
// into gv and, at a spring's first end, dJ/dks into gks.  Every spring is
// evaluated from this vertex's side, which is bitwise the negated terms of
// the other side, so it is always added.  constants(k, sp, L0, ks, kd) reads
// a spring's.  What bounds it is the chain slot -> neighbour and constants ->
// terms, so slots are read two springs ahead, neighbours and constants one,
// by unconditional loads (of vertex i itself past the last slot).
template <class Constants>
__device__ __forceinline__ void adj_gather_springs(const AdjGatherIn& c, int i, int nx, float h, float hh,
                                                   const Constants& constants, float* gks, V3& gx, V3& gv) {
    if (c.wa < 1) return;
    const int N = c.N;
    struct Slot {
        int sp;
        uint16_t m;
    };
    struct Spring {
        int sp;
        bool second;
        V3 x, v, mu, p;
        float L0, ks, kd, g;
    };
    auto slot = [&](int k) {
        const size_t o = (size_t)min(k, c.wa - 1) * N + i;
        Slot r = {c.ainc_s[o], c.ainc_m[o]};
        if (k >= c.wa) r.sp = -1;
        return r;
    };
    auto fetch = [&](int k, Slot q) {
        const bool have = q.sp >= 0;
        Spring r;
        r.sp = q.sp;
        r.second = (q.m >> 8) & 1u;
        const int j = have ? i + slot_dj(q.m) * nx + slot_di(q.m) : i, sp = have ? q.sp : 0;
        r.x = ld3(c.x, N, j);
        r.v = ld3(c.v, N, j);
        r.mu = ld3(c.mu, N, j);
        r.p = ld3(c.p, N, j);
        constants(min(k, c.wa - 1), sp, r.L0, r.ks, r.kd);
        r.g = gks[r.second ? 0 : sp];  // (the first end adds; the ids of a column are far apart)
        return r;
    };
    const V3 xi = ld3(c.x, N, i), vi = ld3(c.v, N, i), mi = ld3(c.mu, N, i), pi = ld3(c.p, N, i);
    const V3 wi = add3(vi, pi);
    Slot ahead = slot(1);
    Spring nxt = fetch(0, slot(0));
#pragma unroll 1
    for (int k = 0; k < c.wa; k++) {
        const Spring in = nxt;
        if (in.sp < 0) break;
        const Slot q = ahead;
        ahead = slot(k + 2);
        nxt = fetch(k + 1, q);
        float ge[3], gvv[3], gk;
        spring_adjoint(xi, in.x, vi, in.v, mi, in.mu, wi, add3(in.v, in.p), pi, in.p, in.L0, in.ks, in.kd, h, hh, ge,
                       gvv, gk);
        gx = {gx.x + ge[0], gx.y + ge[1], gx.z + ge[2]};
        gv = {gv.x + gvv[0], gv.y + gvv[1], gv.z + gvv[2]};
        if (!in.second) gks[in.sp] = in.g + gk;
    }
}

}  // namespace dev
}  // namespace oc
