// Post-step passes of StepPhysics and the position-Verlet step (gfx950).
//
//   k_ellipsoid : EllipsoidCollision (IE:727-751, VL:509-533), per vertex
//   k_provot    : ApplyProvotDynamicInverse (IE:702-726), per-vertex gather
//                 of the springs' velocity corrections in list order (the
//                 reference only reads X there, so the gather equals its
//                 sequential scatter bit for bit)
//   k_verlet    : ComputeForces(dt) + IntegrateVerlet (VL:428-484) fused per
//                 vertex on 32x8 tiles, whose positions and velocities (with
//                 a 2-wide halo) are staged in LDS; reads x, x_last and
//                 writes the next positions into a third buffer, so no
//                 thread sees a half-updated neighbour
//
// Expressions follow the reference's GLM order, built with -ffp-contract=off.
#include <algorithm>

#include "oc_device.hpp"

namespace oc {

namespace {

using namespace dev;

__global__ __launch_bounds__(256) void k_ellipsoid(float* x, float* w, int N, oc_ellipsoid e,
                                                   int mode) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= N) return;
    const V3 p = ld3(x, N, i);
    bool inside;
    const V3 q = ellipsoid_push(e, p, inside);
    if (!inside) return;
    st3(x, N, i, q);
    st3(w, N, i, mode == 1 ? q : V3{0.0f, 0.0f, 0.0f});
}

// Velocity correction of one spring for its endpoints (IE:706-714).
__device__ inline bool provot_delta(V3 x1, V3 x2, float rest, float slack, V3& dP) {
    V3 dp = sub3(x1, x2);
    const float sq = dp.x * dp.x + dp.y * dp.y + dp.z * dp.z;
    float dist = sqrtf(sq);
    const float thr = rest * slack;
    if (!(dist > thr)) return false;
    dist -= thr;
    dist /= 2.0f;
    const float inv = 1.0f / sqrtf(sq);
    dP = {(dp.x * inv) * dist, (dp.y * inv) * dist, (dp.z * inv) * dist};
    return true;
}

// A vertex's corrections in slot order.  The slot table is read three springs
// ahead, the other end's position and pin and the rest length two, in a loop
// of 1 KB: with every load of every slot issued first the code was 20 KB,
// straight through, and a launch spends about 0.4 us per KB on fetching code
// that it runs once.  21x21: 10.8 -> 9 us.
constexpr int kProvotThreads = 64;
__global__ __launch_bounds__(kProvotThreads) void k_provot(DevCloth c, float slack) {
    const int i = blockIdx.x * kProvotThreads + threadIdx.x;
    if (i >= c.N) return;
    const int N = c.N;
    struct Slot {
        int sp;
        uint16_t m;
    };
    struct Spring {
        int sp;
        uint16_t m;
        V3 x;
        float rest;
        bool pin;
    };
    auto slot = [&](int k) {
        const size_t o = (size_t)min(k, c.wa - 1) * N + i;
        Slot r = {c.ainc_s[o], c.ainc_m[o]};
        if (k >= c.wa) r.sp = -1;
        return r;
    };
    auto fetch = [&](Slot q) {  // of vertex i itself past the last slot
        const int j = q.sp >= 0 ? i + slot_dj(q.m) * c.nx + slot_di(q.m) : i;
        return Spring{q.sp, q.m, ld3(c.x, N, j), c.L0[max(q.sp, 0)], c.pin[j] != 0};
    };
    if (c.wa < 1) return;
    const Slot s0 = slot(0), s1 = slot(1);
    Slot ahead = slot(2);
    Spring nxt = fetch(s0), nxt2 = fetch(s1);
    const V3 xi = ld3(c.x, N, i);
    V3 v = ld3(c.v, N, i);
    const bool pin_i = c.pin[i] != 0;
    bool touched = false;
#pragma unroll 1
    for (int k = 0; k < c.wa; k++) {
        const Spring in = nxt;
        if (in.sp < 0) break;  // (the slots are packed)
        const Slot q = ahead;
        ahead = slot(k + 3);
        nxt = nxt2;
        nxt2 = fetch(q);
        const bool second = (in.m >> 8) & 1u;
        V3 dP;  // from the first end's side
        const V3 a = second ? in.x : xi, b = second ? xi : in.x;
        if (!provot_delta(a, b, in.rest, slack, dP)) continue;
        if (!second) {  // i is p1: V[p1] -= dP unless p1 is pinned
            if (!pin_i) {
                v = sub3(v, dP);
                touched = true;
            }
        } else if (in.pin || !pin_i) {  // i is p2: V[p2] += dP when p1 is pinned or p2 is free
            v = add3(v, dP);
            touched = true;
        }
    }
    if (touched) st3(c.v, N, i, v);
}

// Verlet step on a 2D tile with a kHalo-wide halo staged in LDS: positions
// and Verlet velocities v = (x - x_last)/dt of the window are computed once
// (the same division per vertex as evaluating them per spring end).
template <int TX, int TY>
struct VerletShared {
    static constexpr int WX = TX + 2 * kHalo, WY = TY + 2 * kHalo;
    float wx[3][WY][WX];
    float wv[3][WY][WX];
};

// A vertex's next position (VL:428-444).
__device__ __forceinline__ V3 verlet_next(const VerletScalars& s, V3 xi, V3 xl, V3 F) {
    const float c2 = (s.dt * s.dt) / s.mass;
    V3 xn = {xi.x + (xi.x - xl.x) + c2 * F.x, xi.y + (xi.y - xl.y) + c2 * F.y, xi.z + (xi.z - xl.z) + c2 * F.z};
    if ((s.flags & OC_FLAG_GROUND_CLAMP) && xn.y < 0.0f) xn.y = 0.0f;
    return xn;
}

// Force on vertex t of a tile (VL:448-484): gravity on free vertices, damping
// on all, springs in list order (pinned vertices: damping only).  Springs are
// evaluated from this vertex's side (x1 = x_i), which is bitwise the negated
// p1-side force, so it is always added.  out(i, x_i, F) takes it; a tile past
// the last has no vertices.
// STENCIL: the topology has the stencil assembly form; a vertex's springs
// come from its ownership mask in stencil order (the slot order on such
// topologies) and their constants from the owner planes at the pair's lower
// vertex, so no slot table or spring-id gather is read.
template <int TX, int TY, int WA, bool STENCIL, class Out>
__device__ __forceinline__ void verlet_tile(const DevVerlet& c, const VerletScalars& s, VerletShared<TX, TY>& sh, int tile,
                                            int t, const Out& out) {
    constexpr int NT = TX * TY, H = kHalo;
    constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    constexpr int NWIN = (WX * WY + NT - 1) / NT;
    const int ntx = (c.nx + TX - 1) / TX;
    const int bx = tile % ntx, by = tile / ntx;
    const int lx = t % TX, ly = t / TX;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int N = c.N, i = gj * c.nx + gi;
    int sps[WA];
    uint16_t ms[WA];
    uint32_t mi = 0u;
    if constexpr (STENCIL) {
        mi = own ? c.asm_mask[i] : 0u;
    } else {
#pragma unroll
        for (int k = 0; k < WA; k++) {
            sps[k] = (own && k < c.wa) ? c.ainc_s[k * N + i] : -1;
            ms[k] = (own && k < c.wa) ? c.ainc_m[k * N + i] : kEmptySlot;
        }
    }
    const int x0 = bx * TX - H, y0 = by * TY - H;
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = t + n * NT;
        if (idx < WX * WY) {
            const int wx = idx % WX, wy = idx / WX;
            const int gx = x0 + wx, gy = y0 + wy;
            V3 xw = {0.0f, 0.0f, 0.0f}, vw = xw;
            if (gx >= 0 && gx < c.nx && gy >= 0 && gy < c.ny) {
                const int g = gy * c.nx + gx;
                xw = ld3(c.x, N, g);
                const V3 xl = ld3(c.xl, N, g);
                vw = {(xw.x - xl.x) / s.dt, (xw.y - xl.y) / s.dt, (xw.z - xl.z) / s.dt};
            }
            sh.wx[0][wy][wx] = xw.x;
            sh.wx[1][wy][wx] = xw.y;
            sh.wx[2][wy][wx] = xw.z;
            sh.wv[0][wy][wx] = vw.x;
            sh.wv[1][wy][wx] = vw.y;
            sh.wv[2][wy][wx] = vw.z;
        }
    }
    __syncthreads();
    if (!own) return;
    const int cy = ly + H, cx = lx + H;
    const V3 xi = {sh.wx[0][cy][cx], sh.wx[1][cy][cx], sh.wx[2][cy][cx]};
    const V3 vi = {sh.wv[0][cy][cx], sh.wv[1][cy][cx], sh.wv[2][cy][cx]};
    const bool pinned = c.pin[i] != 0;
    V3 F = {0.0f, 0.0f, 0.0f};
    if (!pinned) F = {F.x + s.gx * s.mass, F.y + s.gy * s.mass, F.z + s.gz * s.mass};
    F = {F.x + s.damping * vi.x, F.y + s.damping * vi.y, F.z + s.damping * vi.z};
    if (!pinned && STENCIL) {
#pragma unroll
        for (int k = 0; k < kStencil; k++) {
            if (!((mi >> k) & 1u)) continue;
            const int wy = cy + stencil_dj(k), wx = cx + stencil_di(k);
            const V3 xj = {sh.wx[0][wy][wx], sh.wx[1][wy][wx], sh.wx[2][wy][wx]};
            const V3 vj = {sh.wv[0][wy][wx], sh.wv[1][wy][wx], sh.wv[2][wy][wx]};
            const int g = stencil_owner(k) ? i : i + stencil_dj(k) * c.nx + stencil_di(k);
            const float* cp = c.cst + (size_t)owned_index(k) * 3 * N + g;
            F = add3(F, spring_force(xi, xj, vi, vj, cp[0], cp[N], cp[2 * (size_t)N]));
            if ((mi >> (16 + k)) & 1u) {  // the pair's second spring (multiplicity 1 planes)
                const float* c2 = cp + (size_t)kOwned * 3 * N;
                F = add3(F, spring_force(xi, xj, vi, vj, c2[0], c2[N], c2[2 * (size_t)N]));
            }
        }
    } else if (!pinned) {
#pragma unroll
        for (int k = 0; k < WA; k++) {
            const int sp = sps[k];
            if (sp < 0) break;
            const int wy = cy + slot_dj(ms[k]), wx = cx + slot_di(ms[k]);
            const V3 xj = {sh.wx[0][wy][wx], sh.wx[1][wy][wx], sh.wx[2][wy][wx]};
            const V3 vj = {sh.wv[0][wy][wx], sh.wv[1][wy][wx], sh.wv[2][wy][wx]};
            F = add3(F, spring_force(xi, xj, vi, vj, c.L0[sp], c.ks[sp], c.kd[sp]));
        }
    }
    out(i, xi, F);
}

// One step of all vertices, or (FORCES) their forces.
template <int TX, int TY, int WA, bool FORCES, bool STENCIL>
__global__ __launch_bounds__(TX* TY) void k_verlet(DevVerlet c, VerletScalars s) {
    __shared__ VerletShared<TX, TY> sh;
    const int nt = ((c.nx + TX - 1) / TX) * ((c.ny + TY - 1) / TY);
    verlet_tile<TX, TY, WA, STENCIL>(c, s, sh, tile_of_block(blockIdx.x, nt), threadIdx.x, [&](int i, V3 xi, V3 F) {
        if constexpr (FORCES)
            st3(c.f, c.N, i, F);
        else
            st3(c.xn, c.N, i, verlet_next(s, xi, ld3(c.xl, c.N, i), F));
    });
}

// The Verlet step has no reduction, so its tile shape is free: 32x8 measured
// faster than the implicit kernels' 64x8 at 512x512 (15.5 against 17.4 us).
constexpr int kVerletTileX = 32, kVerletTileY = 8;

// ---------------------------------------------------------------------------
// resident Verlet: many steps in one launch, the cloth in registers and LDS
// ---------------------------------------------------------------------------
// A launch per step reads 36 floats of every vertex and its springs again and
// waits for the launch before it.  Here every block keeps a region of T x T
// vertices for all steps of a call, a vertex per thread: positions and spring
// constants in registers, the region's positions and velocities with their
// halo in LDS.  In a step a thread evaluates the six springs its vertex owns
// (threads of the first waves also one of the strips around the region, whose
// owners are outside), hands the forces to the partners through LDS, and adds
// all of its vertex's in stencil order.  The outer two rows and columns go to
// the neighbouring regions as 8-byte words (value, tag) that are stored and
// polled with relaxed device-scope accesses, each its own flag.  A region
// publishes step n + 2 only after it has read its neighbours' step n + 1, and
// these publish that only after they have read its step n, so two sets of
// words are enough.  The tag's low bit tells that the collider moved the
// vertex (its previous position is then the position itself; else the reader
// knows it).  Blocks wait for each other, so all must run: there is one per CU
// at most, and they call the roll first.  Where other work holds CUs for too
// long, the roll is closed and every block, those that start later too, takes
// tiles of whole steps in memory by tickets, so the steps are done in any case.
// After a complete roll every wait ends; each is bounded all the same, and one
// that ends without its word sets *err and every block leaves.
//
// Measured per step of 200, with the collider, a launch each for step and
// collider before: 512x512 14.2 -> 6.3 us, 256x256 12 -> 4.5, 21x21 8.4 ->
// 3.6.  About 1 us of it is the exchange; the rest is the chain through a step
// (six springs with a square root and two divisions each, the sum over
// twelve, three barriers), at 512x512 with four waves per SIMD to issue (635
// vector instructions per wave and step, 69% of the issue slots).
constexpr int kVerletPolls = 1 << 21;  // seconds

template <int T>
struct VerletRegion {
    static constexpr int NT = T * T, H = kHalo, W = T + 2 * H, NW = W * W, NS = strip_total<T, T>();
    static constexpr int NH = NW - NT;  // halo vertices
    static constexpr int HR = (3 * NH + NT - 1) / NT;
    static constexpr int NJ = NT - NS;  // second springs a region can take (see below)
    static constexpr size_t lds = sizeof(float) * (6 * NW + 18 * NT + 3 * NT);
};

// What steps by tickets take: the arguments of k_verlet_resident again, as
// arguments of their own.  (Shared, they stay in scalar registers from the
// kernel's start, and what a resident step needs is moved out of them.)
struct VerletTickets {
    DevVerlet c;
    VerletScalars s;
    float* x;
    float* xl;
    oc_ellipsoid e;
    int has_e, nsteps;
    unsigned* q;
};

// The steps by tickets, G tiles per ticket (a thread per vertex), from the
// state x, xl to c.xn, c.f and back; after an odd number a last phase copies.
template <int T>
__device__ inline void verlet_tickets(const VerletTickets& a, float* lds, Ticket& t) {
    constexpr int TX = kVerletTileX, TY = kVerletTileY, G = T * T / (TX * TY);
    static_assert(G >= 1 && G * sizeof(VerletShared<TX, TY>) <= VerletRegion<T>::lds, "a window per tile");
    VerletShared<TX, TY>* const sh = reinterpret_cast<VerletShared<TX, TY>*>(lds) + threadIdx.x / (TX * TY);
    const int nt = ((a.c.nx + TX - 1) / TX) * ((a.c.ny + TY - 1) / TY), N = a.c.N;
    const unsigned pieces = (unsigned)(nt + G - 1) / G, total = (unsigned)(a.nsteps + (a.nsteps & 1)) * pieces;
    while (ticket_take(a.q, pieces, total, nullptr, a.c.err, t) == kTicketWork) {
        const int n = (int)(t.n / pieces), tile = (int)(t.n % pieces) * G + (int)threadIdx.x / (TX * TY);
        const bool odd = n & 1;
        DevVerlet d = a.c;
        d.x = odd ? a.c.xn : a.x;
        d.xl = odd ? a.c.f : a.xl;
        float* const to = odd ? a.x : a.c.xn;
        float* const tol = odd ? a.xl : a.c.f;
        verlet_tile<TX, TY, 1, true>(d, a.s, *sh, tile, threadIdx.x % (TX * TY), [&](int i, V3 xi, V3 F) {
            V3 p = xi, last = ld3(d.xl, N, i);
            if (n < a.nsteps) {
                bool moved = false;
                p = verlet_next(a.s, xi, last, F);
                if (a.has_e) p = ellipsoid_push(a.e, p, moved);
                last = moved ? p : xi;
            }
            st3(to, N, i, p);
            st3(tol, N, i, last);
        });
        ticket_done(a.q);
    }
}

// set: which of the two sets of control words (c.sync) this launch uses; it
// clears the other, which the launch before has left.  nb: the regions.
template <int T>
__global__ __launch_bounds__(T* T) void k_verlet_resident(DevVerlet c, VerletScalars s, float* xo, float* xlo, int nsteps,
                                                          unsigned base, oc_ellipsoid e, int has_e, int set, int nb,
                                                          VerletTickets rest) {
    using R = VerletRegion<T>;
    constexpr int NT = R::NT, H = R::H, W = R::W, NW = R::NW, NS = R::NS;
    static_assert(R::NJ > 0 && 4 * R::NJ <= 18 * NT, "one extra spring per thread, room for their list");
    extern __shared__ float lds[];
    __shared__ int lost, jobs, all;
    __shared__ Ticket ticket;
    unsigned* const ctl = c.sync + set * kSyncWords;
    if (threadIdx.x == 0) {
        roll_call_sign(ctl + 1);
        unsigned* const other = c.sync + (1 - set) * kSyncWords;
        if (blockIdx.x == 0) other[1] = other[kSyncTickets] = other[kSyncTickets + kTicketDone] = 0;
    }
    float* const wx = lds;           // 3 planes of the window: positions
    float* const wv = lds + 3 * NW;  // velocities
    float* const fo = lds + 6 * NW;  // 18 planes of NT: force of own spring o, component c at plane 3 o + c
    float* const fs = fo + 18 * NT;  // 3 planes of NT: the threads' extra springs' forces
    const int tid = threadIdx.x, N = c.N, nx = c.nx, ny = c.ny;
    const int ntx = (nx + T - 1) / T, nt = ntx * ((ny + T - 1) / T);
    const int tile = tile_of_block(blockIdx.x, nt);
    const int bx = tile % ntx, by = tile / ntx;
    const int lx = tid % T, ly = tid / T;
    const int gi = bx * T + lx, gj = by * T + ly, i = gj * nx + gi;
    const bool own = gi < nx && gj < ny;
    if (tid == 0) lost = jobs = 0;
    for (int w = tid; w < NW; w += NT) {
        const int gx = bx * T - H + w % W, gy = by * T - H + w / W;
        V3 x = {0.0f, 0.0f, 0.0f}, v = x;
        if (gx >= 0 && gx < nx && gy >= 0 && gy < ny) {
            x = ld3(c.x, N, gy * nx + gx);
            const V3 xl = ld3(c.xl, N, gy * nx + gx);
            v = {(x.x - xl.x) / s.dt, (x.y - xl.y) / s.dt, (x.z - xl.z) / s.dt};
        }
        wx[w] = x.x;
        wx[NW + w] = x.y;
        wx[2 * NW + w] = x.z;
        wv[w] = v.x;
        wv[NW + w] = v.y;
        wv[2 * NW + w] = v.z;
    }
    const int at = (ly + H) * W + lx + H;
    V3 xi = {0.0f, 0.0f, 0.0f}, xl = xi;
    uint32_t mi = 0u;
    bool pinned = true;
    float L0[kOwned], ks[kOwned], kd[kOwned];
#pragma unroll
    for (int o = 0; o < kOwned; o++) L0[o] = ks[o] = kd[o] = 0.0f;
    if (own) {
        xi = ld3(c.x, N, i);
        xl = ld3(c.xl, N, i);
        mi = c.asm_mask[i];
        pinned = c.pin[i] != 0;
#pragma unroll
        for (int o = 0; o < kOwned; o++) {
            const float* p = c.cst + (size_t)(3 * o) * N + i;
            L0[o] = p[0];
            ks[o] = p[N];
            kd[o] = p[2 * (size_t)N];
        }
    }
    // this thread's extra spring: the window places of its ends, -1 for none.
    // The first threads' are the strips'; the next ones' the second springs
    // of the region's pairs (the stencil's duplicated bends), which each end
    // evaluates for itself: a vertex lists its own, at most two (second), in
    // stencil order
    int sa = -1, sb = 0;
    float sL0 = 0.0f, sks = 0.0f, skd = 0.0f;
    if (tid < NS) {
        int o, k, px, py;
        strip_of_column<T, T>(tid, o, k);
        strip_owner<T, T>(o, k, px, py);
        const int gx = bx * T + px, gy = by * T + py;
        if (gx >= 0 && gx < nx && gy >= 0 && gy < ny && ((c.asm_mask[gy * nx + gx] >> owned_k(o)) & 1u)) {
            const float* p = c.cst + (size_t)(3 * o) * N + gy * nx + gx;
            sL0 = p[0];
            sks = p[N];
            skd = p[2 * (size_t)N];
            sa = (py + H) * W + px + H;
            sb = sa + own_dy(o) * W + own_dx(o);
        }
    }
    __syncthreads();
    unsigned second = 0;
    {
        int found = 0;
#pragma unroll 1
        for (unsigned m = mi >> 16; m; m &= m - 1u) {
            const int k = __ffs(m) - 1, o = owned_index(k);
            const int slot = atomicAdd(&jobs, 1);
            if (slot >= R::NJ || found >= 2) break;  // (verlet_seconds_fit has ruled this out)
            const float* p = c.cst + (size_t)(3 * (kOwned + o)) * N +
                             (stencil_owner(k) ? i : i + stencil_dj(k) * nx + stencil_di(k));
            float* const job = fo + 4 * slot;
            job[0] = __int_as_float(at | (at + stencil_dj(k) * W + stencil_di(k)) << 16);
            job[1] = p[0];
            job[2] = p[N];
            job[3] = p[2 * (size_t)N];
            second |= (unsigned)(NS + slot) << (16 * found++);
        }
    }
    __syncthreads();
    if (tid >= NS && tid - NS < jobs) {
        const float* job = fo + 4 * (tid - NS);
        sa = __float_as_int(job[0]) & 0xFFFF;
        sb = __float_as_int(job[0]) >> 16;
        sL0 = job[1];
        sks = job[2];
        skd = job[3];
    }
    // where the force of the partner's spring in direction o is: in fo, or
    // (one's complement) in fs
    int part[kOwned];
#pragma unroll
    for (int o = 0; o < kOwned; o++) {
        const int px = lx - own_dx(o), py = ly - own_dy(o);
        part[o] = px >= 0 && px < T && py >= 0 && py < T ? 3 * o * NT + py * T + px
                                                         : ~(strip_base<T, T>(o) + strip_index<T, T>(o, px, py));
    }
    // the halo words this thread reads: word of the exchange (-1: outside the
    // cloth) and place in the window's planes
    int hsrc[R::HR], hdst[R::HR];
#pragma unroll
    for (int q = 0; q < R::HR; q++) {
        const int k = tid + q * NT, h = k / 3, comp = k % 3;
        int px = 0, py = 0;
        if (h < 2 * W) {
            px = h % W;
            py = h / W;
        } else if (h < 4 * W) {
            px = h % W;
            py = T + h / W;
        } else {
            const int r = h - 4 * W;
            px = (r & 1) + (r >= 2 * T ? T + H : 0);
            py = H + (r % (2 * T)) / 2;
        }
        const int gx = bx * T - H + px, gy = by * T - H + py;
        hsrc[q] = h < R::NH && gx >= 0 && gx < nx && gy >= 0 && gy < ny ? 4 * (gy * nx + gx) + comp : -1;
        hdst[q] = comp * NW + py * W + px;
    }
    const bool rim = own && (lx < H || lx >= T - H || ly < H || ly >= T - H);
    auto win = [&](const float* p, int a) { return V3{p[a], p[NW + a], p[2 * NW + a]}; };

    if (tid == 0) all = roll_call_wait(ctl + 1, nb);
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(all)) {
        verlet_tickets<T>(rest, lds, ticket);
        return;
    }

    // What the steps take from outside is too much for the scalar registers.
    // One wave per SIMD (T = 16) loses least by testing the mask's bits anew
    // (here) and loading the collider's numbers in every step: 21x21 3.62 us a
    // step, 3.71 with the bits' 24 conditions and the numbers kept and spilled;
    // with four (T = 32), it is the other way round: 512x512 6.44 and 6.35.
    oc_ellipsoid ball = e;
    if constexpr (T == 32) {
#pragma unroll
        for (int k = 0; k < 16; k++)
            if (k % 4 < 3) asm volatile("" : "+s"(ball.inverse[k]));
#pragma unroll
        for (int k = 0; k < 3; k++) asm volatile("" : "+s"(ball.center[k]));
    }
    for (int n = 0; n < nsteps; n++) {
        __syncthreads();  // the window is complete
        if (lost) return;
        const V3 vi = win(wv, at);
        V3 f[kOwned];
#pragma unroll
        for (int o = 0; o < kOwned; o++) {
            const int b = at + own_dy(o) * W + own_dx(o);  // (without a pair: not used)
            f[o] = spring_force(xi, win(wx, b), vi, win(wv, b), L0[o], ks[o], kd[o]);
            fo[(3 * o) * NT + tid] = f[o].x;
            fo[(3 * o + 1) * NT + tid] = f[o].y;
            fo[(3 * o + 2) * NT + tid] = f[o].z;
        }
        if (sa >= 0) {
            const V3 g = spring_force(win(wx, sa), win(wx, sb), win(wv, sa), win(wv, sb), sL0, sks, skd);
            fs[tid] = g.x;
            fs[NT + tid] = g.y;
            fs[2 * NT + tid] = g.z;
        }
        __syncthreads();
        V3 F = {0.0f, 0.0f, 0.0f};
        if (!pinned) F = {F.x + s.gx * s.mass, F.y + s.gy * s.mass, F.z + s.gz * s.mass};
        F = {F.x + s.damping * vi.x, F.y + s.damping * vi.y, F.z + s.damping * vi.z};
        if (!pinned) {
            unsigned q = second;
            const unsigned bits = T == 16 ? here(mi) : mi;
#pragma unroll
            for (int k = 0; k < kStencil; k++) {
                if (!((bits >> k) & 1u)) continue;
                const int o = owned_index(k);
                if (stencil_owner(k)) {
                    F = add3(F, f[o]);
                } else {  // the force on the spring's owner
                    const float* p = part[o] >= 0 ? fo + part[o] : fs + ~part[o];
                    F = sub3(F, V3{p[0], p[NT], p[2 * NT]});
                }
                if ((bits >> (16 + k)) & 1u) {
                    const float* p = fs + (q & 0xFFFFu);
                    F = add3(F, V3{p[0], p[NT], p[2 * NT]});
                    q >>= 16;
                }
            }
        }
        V3 xn = verlet_next(s, xi, xl, F);
        xl = xi;
        bool moved = false;
        if (has_e) xn = ellipsoid_push(ball, xn, moved);
        if (moved) xl = xn;
        xi = xn;
        if (n + 1 == nsteps) break;
        uint64_t* const words = c.xch + (size_t)(n & 1) * 4 * N;
        const unsigned tag = base + 2u * (unsigned)(n + 1);
        if (rim) {
            xch_store(words, 4u * i, tag + moved, xi.x);
            xch_store(words, 4u * i + 1u, tag + moved, xi.y);
            xch_store(words, 4u * i + 2u, tag + moved, xi.z);
        }
        __syncthreads();  // the window has been read
        wx[at] = xi.x;
        wx[NW + at] = xi.y;
        wx[2 * NW + at] = xi.z;
        wv[at] = (xi.x - xl.x) / s.dt;
        wv[NW + at] = (xi.y - xl.y) / s.dt;
        wv[2 * NW + at] = (xi.z - xl.z) / s.dt;
#pragma unroll
        for (int q = 0; q < R::HR; q++) {
            if (hsrc[q] < 0) continue;
            uint64_t w = xch_load(words, (unsigned)hsrc[q]);
            for (int polls = 0; (((unsigned)(w >> 32)) & ~1u) != tag; polls++) {
                if (polls == kVerletPolls) {
                    lost = 1;
                    __hip_atomic_store(c.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    break;
                }
                w = xch_load(words, (unsigned)hsrc[q]);
            }
            const float x = __uint_as_float((unsigned)w), before = ((w >> 32) & 1u) ? x : wx[hdst[q]];
            wx[hdst[q]] = x;
            wv[hdst[q]] = (x - before) / s.dt;
        }
    }
    if (own) {
        st3(xo, N, i, xi);
        st3(xlo, N, i, xl);
    }
}

template <bool FORCES>
hipError_t launch_verlet(const DevVerlet& c, const VerletScalars& s, hipStream_t st) {
    constexpr int TX = kVerletTileX, TY = kVerletTileY;
    const int nt = ((c.nx + TX - 1) / TX) * ((c.ny + TY - 1) / TY);
    if (c.stencil_asm)
        hipLaunchKernelGGL((k_verlet<TX, TY, 1, FORCES, true>), dim3(nt), dim3(TX * TY), 0, st, c, s);
    else if (c.wa <= 16)
        hipLaunchKernelGGL((k_verlet<TX, TY, 16, FORCES, false>), dim3(nt), dim3(TX * TY), 0, st, c, s);
    else
        hipLaunchKernelGGL((k_verlet<TX, TY, kMaxAssemblyWidth, FORCES, false>), dim3(nt), dim3(TX * TY), 0,
                           st, c, s);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_ellipsoid(float* x, float* w, int N, const oc_ellipsoid& e, int mode,
                            hipStream_t st) {
    hipLaunchKernelGGL(k_ellipsoid, dim3((N + 255) / 256), dim3(256), 0, st, x, w, N, e, mode);
    return hipGetLastError();
}

hipError_t launch_provot(const DevCloth& c, float slack, hipStream_t st) {
    hipLaunchKernelGGL(k_provot, dim3((c.N + kProvotThreads - 1) / kProvotThreads), dim3(kProvotThreads), 0, st, c, slack);
    return hipGetLastError();
}

// CUs, if a region's block fits one.
template <int T>
static int verlet_blocks_fit() {
    int dev = 0, cus = 0, per_cu = 0, lds = 0;
    if (!hip_ok(hipGetDevice(&dev)) || !hip_ok(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) ||
        !hip_ok(hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) ||
        VerletRegion<T>::lds + 64 > (size_t)lds ||
        !hip_ok(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_verlet_resident<T>, T * T, VerletRegion<T>::lds)))
        return 0;
    return per_cu > 0 ? cus : 0;
}

static int verlet_regions(int nx, int ny, int T) { return ((nx + T - 1) / T) * ((ny + T - 1) / T); }

// A region's second springs have a thread each, a vertex at most two.
template <int T>
static bool verlet_seconds_fit(int nx, int ny, const uint32_t* mask) {
    for (int by = 0; by < ny; by += T)
        for (int bx = 0; bx < nx; bx += T) {
            int n = 0;
            for (int y = by; y < std::min(by + T, ny); y++)
                for (int x = bx; x < std::min(bx + T, nx); x++) {
                    const int k = __builtin_popcount(mask[(size_t)y * nx + x] >> 16);
                    if (k > 2) return false;
                    n += k;
                }
            if (n > VerletRegion<T>::NJ) return false;
        }
    return true;
}

// The smaller regions while each has a CU of its own (a wave per SIMD: 256x256
// 4.5 us per step, in 32x32 regions 5.2; 128x128 3.8 and 5.2), then the larger
// ones (512x512 6.3 us, in 1024 small regions, four per CU, 7.0).
int verlet_resident_region(int nx, int ny, const uint32_t* mask) {
    if (verlet_regions(nx, ny, 16) <= verlet_blocks_fit<16>() && verlet_seconds_fit<16>(nx, ny, mask)) return 16;
    if (verlet_regions(nx, ny, 32) <= verlet_blocks_fit<32>() && verlet_seconds_fit<32>(nx, ny, mask)) return 32;
    return 0;
}

hipError_t launch_verlet_resident(const DevVerlet& c, const VerletScalars& s, float* x, float* xl, int T, int nsteps,
                                  unsigned base, int set, const oc_ellipsoid* e, int blocks, hipStream_t st) {
    const int nb = verlet_regions(c.nx, c.ny, T == 16 ? 16 : 32);
    if ((T != 16 && T != 32) || nsteps < 2 || nsteps > kVerletMost || (base & 1u) || !c.stencil_asm || x != c.x ||
        xl != c.xl || (set & ~1) || blocks < 0 || blocks > nb)
        return hipErrorInvalidValue;
    const oc_ellipsoid el = e ? *e : oc_ellipsoid{};
    const dim3 grid(blocks ? blocks : nb), block(T * T);
    const VerletTickets rest = {c, s, x, xl, el, e != nullptr, nsteps, c.sync + set * kSyncWords + kSyncTickets};
    if (T == 16)
        hipLaunchKernelGGL(k_verlet_resident<16>, grid, block, VerletRegion<16>::lds, st, c, s, x, xl, nsteps, base, el,
                           e != nullptr, set, nb, rest);
    else
        hipLaunchKernelGGL(k_verlet_resident<32>, grid, block, VerletRegion<32>::lds, st, c, s, x, xl, nsteps, base, el,
                           e != nullptr, set, nb, rest);
    return hipGetLastError();
}

hipError_t launch_verlet_forces(const DevVerlet& c, const VerletScalars& s, hipStream_t st) {
    return launch_verlet<true>(c, s, st);
}

hipError_t launch_verlet_step(const DevVerlet& c, const VerletScalars& s, hipStream_t st) {
    return launch_verlet<false>(c, s, st);
}

}  // namespace oc
