// HIP kernels of the implicit mass-spring step (gfx950, wave64).
//
// One step (OpenCloth_ImplicitEuler/.../main.cpp:774-779 without the
// post-step passes) is
//   assemble  : per-vertex gather of spring forces and 3x3 Jacobian blocks,
//               rhs b = h(f + h df/dx v), pair blocks C, CG start r = S(b - A dv)
//   cg_spmv   : d = r + beta d on the tile and its halo in LDS, q = S A d,
//               partial d.q                                    (x iterations)
//   cg_axpy   : dv += alpha d, r -= alpha q, partial r.r        (x iterations)
//   cg_finish : iteration count and status
//   update    : v += dv, x += h v
//
// Layout: vertex vectors are SoA planes (x[c*N + i]).  Pair blocks live in
// planes: the block of the pair (a, b = a + offset_p) is stored at
// blocks[(p*6 + comp)*N + a], so neighbouring threads read neighbouring
// addresses for every stencil direction.  The diagonal block
// A_ii = m I - sum_j C_ij is never stored: (A d)_i = m d_i + sum_j C_ij (d_j - d_i).
//
// Arithmetic follows the reference's GLM expression order with no FMA
// contraction (built with -ffp-contract=off), so per-spring forces and blocks
// equal the CPU oracle bit for bit.  Reductions use one fixed tree: a 64-lane
// shuffle tree per wave, the waves of a tile in order, then a lane-strided
// pass over tile partials followed by the same lane tree.  Partials are
// indexed by tile, so the block-to-tile mapping does not change any sum.
//
// Every CG kernel issues all loads that do not depend on the previous
// reduction (its own vectors, pair blocks, the partials) before waiting, so
// the cross-tile reduction overlaps the memory traffic.
#include <hip/hip_ext.h>

#include <algorithm>

#include "oc_device.hpp"
#include "cg_control.hpp"

namespace oc {

namespace {

constexpr int H = kHalo;
using namespace dev;


// Jacobi preconditioner entry 1/diag(A); a non-positive or non-finite
// diagonal (A can be indefinite under strong compression) falls back to 1.
__device__ inline float jacobi_inv(float dg) {
    return (dg > 0.0f && isfinite(dg)) ? 1.0f / dg : 1.0f;
}

// ---------------------------------------------------------------------------
// forces (ComputeForces, IE:645-682): gather in spring order, pins get zero
// ---------------------------------------------------------------------------
template <int TX, int TY>
__global__ __launch_bounds__(TX* TY) void k_forces(DevCloth c, StepScalars s) {
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int t = tile_of_block(blockIdx.x, c.nt);
    const int bx = t % c.ntx, by = t / c.ntx;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    if (gi >= c.nx || gj >= c.ny) return;
    const int N = c.N, i = gj * c.nx + gi;
    V3 acc = {0.0f, 0.0f, 0.0f};
    if (!c.pin[i]) {
        V3 xi = ld3(c.x, N, i), vi = ld3(c.v, N, i);
        acc = {0.0f + s.mass * s.gx, 0.0f + s.mass * s.gy, 0.0f + s.mass * s.gz};
        if (s.damp != 0.0f) acc = {acc.x + s.damp * vi.x, acc.y + s.damp * vi.y, acc.z + s.damp * vi.z};
        for (int k = 0; k < c.wa; k++) {
            const int sp = c.ainc_s[k * N + i];
            if (sp < 0) break;
            const uint16_t m = c.ainc_m[k * N + i];
            const int j = i + slot_dj(m) * c.nx + slot_di(m);
            V3 xj = ld3(c.x, N, j), vj = ld3(c.v, N, j);
            const bool second = (m >> 8) & 1u;
            V3 f = second ? spring_force(xj, xi, vj, vi, c.L0[sp], c.ks[sp], c.kd[sp])
                          : spring_force(xi, xj, vi, vj, c.L0[sp], c.ks[sp], c.kd[sp]);
            if (second)
                acc = {acc.x - f.x, acc.y - f.y, acc.z - f.z};
            else
                acc = {acc.x + f.x, acc.y + f.y, acc.z + f.z};
        }
    }
    st3(c.f, N, i, acc);
}

// ---------------------------------------------------------------------------
// assembly + CG start
// ---------------------------------------------------------------------------
// Constants of one incident spring (gathered by spring id).
struct SpringC {
    float L0, ks, kd;
};

template <int WA>
__device__ inline SpringC fetch_constants(const DevCloth& c, const int (&sps)[WA], int k) {
    SpringC r{0.0f, 0.0f, 0.0f};
    const int sp = sps[k];
    if (sp >= 0) {
        r.L0 = ldo(c.L0, (uint32_t)sp);
        r.ks = ldo(c.ks, (uint32_t)sp);
        r.kd = ldo(c.kd, (uint32_t)sp);
    }
    return r;
}

// Tile + halo of x, v and (warm start) dv in LDS.
template <int TX, int TY>
struct AssembleShared {
    static constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    float wx[3][WY][WX];
    float wv[3][WY][WX];
    float wdv[3][WY][WX];
    float ws[TX * TY / 64];
    float bc;
};

// UPD: the window's x and v are the previous step's state before its
// update; apply the update (k_update's arithmetic) on the fly and write the
// tile's updated x, v to xo, vo (other blocks still read x and v).  Only
// with a warm start: a cold start writes dv = 0 here, which other blocks
// would still be reading.
template <int TX, int TY, int WA, bool UPD>
__global__ __launch_bounds__(TX* TY) void k_assemble(DevCloth c, StepScalars s) {
    constexpr int NT = TX * TY;
    constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    constexpr int NWIN = (WX * WY + NT - 1) / NT;
    __shared__ AssembleShared<TX, TY> sh;
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int tile = tile_of_block(blockIdx.x, c.nt);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int N = c.N, i = gj * c.nx + gi;
    if (blockIdx.x == 0) begin_solve<UPD>(c, s, &sh.bc);
    // own slot tables and the first springs' constants, then the window
    int sps[WA];
    uint16_t ms[WA];
#pragma unroll
    for (int k = 0; k < WA; k++) {
        sps[k] = (own && k < c.wa) ? ldo(c.ainc_s, (uint32_t)(k * N + i)) : -1;
        ms[k] = (own && k < c.wa) ? ldo(c.ainc_m, (uint32_t)(k * N + i)) : kEmptySlot;
    }
    constexpr int kPrefetch = 4;
    SpringC pre[kPrefetch];
#pragma unroll
    for (int k = 0; k < kPrefetch; k++) pre[k] = fetch_constants(c, sps, k);
    const int x0 = bx * TX - H, y0 = by * TY - H;
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        if (idx < WX * WY) {
            const int wx = idx % WX, wy = idx / WX;
            const int gx = x0 + wx, gy = y0 + wy;
            V3 xw = {0.0f, 0.0f, 0.0f}, vw = xw, dw = xw;
            if (gx >= 0 && gx < c.nx && gy >= 0 && gy < c.ny) {
                const int g = gy * c.nx + gx;
                xw = ld3o(c.x, N, g);
                vw = ld3o(c.v, N, g);
                if (UPD) {
                    const V3 dp = ld3o(c.dv, N, g);
                    vw = {vw.x + dp.x, vw.y + dp.y, vw.z + dp.z};
                    xw = {xw.x + s.h * vw.x, xw.y + s.h * vw.y, xw.z + s.h * vw.z};
                    if ((s.flags & OC_FLAG_GROUND_CLAMP) && xw.y < 0.0f) xw.y = 0.0f;
                    if (s.warm) dw = dp;
                } else if (s.warm) {
                    dw = ld3o(c.dv, N, g);
                }
            }
            sh.wx[0][wy][wx] = xw.x;
            sh.wx[1][wy][wx] = xw.y;
            sh.wx[2][wy][wx] = xw.z;
            sh.wv[0][wy][wx] = vw.x;
            sh.wv[1][wy][wx] = vw.y;
            sh.wv[2][wy][wx] = vw.z;
            sh.wdv[0][wy][wx] = dw.x;
            sh.wdv[1][wy][wx] = dw.y;
            sh.wdv[2][wy][wx] = dw.z;
        }
    }
    __syncthreads();

    float t = 0.0f;
    if (own) {
        const float h = s.h, hh = s.hh;
        const bool pinned = ldo(c.pin, (uint32_t)i) != 0;
        const int cy = ly + H, cx = lx + H;
        const V3 xi = {sh.wx[0][cy][cx], sh.wx[1][cy][cx], sh.wx[2][cy][cx]};
        const V3 vi = {sh.wv[0][cy][cx], sh.wv[1][cy][cx], sh.wv[2][cy][cx]};
        const V3 dvi = {sh.wdv[0][cy][cx], sh.wdv[1][cy][cx], sh.wdv[2][cy][cx]};
        if (!s.warm) st3o(c.dv, N, i, dvi);
        if (UPD) {
            st3o(c.xo, N, i, xi);
            st3o(c.vo, N, i, vi);
            // k_update's check of the updated state; the bit belongs to the
            // previous step, whose status is already in the sticky word
            if (!(isfinite(xi.x) && isfinite(xi.y) && isfinite(xi.z) && isfinite(vi.x) &&
                  isfinite(vi.y) && isfinite(vi.z)))
                atomicOr(c.ctl + 3, OC_SOLVE_NONFINITE);
        }
        V3 acc = {0.0f, 0.0f, 0.0f}, kv = {0.0f, 0.0f, 0.0f};
        if (!pinned) acc = {0.0f + s.mass * s.gx, 0.0f + s.mass * s.gy, 0.0f + s.mass * s.gz};
        if (!pinned && s.damp != 0.0f)
            acc = {acc.x + s.damp * vi.x, acc.y + s.damp * vi.y, acc.z + s.damp * vi.z};
        V3 adv = {s.md * dvi.x, s.md * dvi.y, s.md * dvi.z};
        V3 dg = {s.md, s.md, s.md};  // diag(A) = m - h c - sum of the pair blocks' diagonals
        float C[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        // Every spring is evaluated from this vertex's side (x1 = x_i): when
        // i is the spring's p2 that negates dp, f and K(v_i - v_j) exactly
        // and leaves K and P unchanged, so adding them equals subtracting
        // the p1-side values bit for bit.  Neighbours come from the LDS
        // window; spring constants are loaded kPrefetch springs ahead.
#pragma unroll
        for (int k = 0; k < WA; k++) {
            const int sp = sps[k];
            if (sp < 0) break;
            const uint16_t m = ms[k];
            const SpringC in = pre[0];
#pragma unroll
            for (int q = 0; q + 1 < kPrefetch; q++) pre[q] = pre[q + 1];
            if (k + kPrefetch < WA) pre[kPrefetch - 1] = fetch_constants(c, sps, k + kPrefetch);
            const int wy = cy + slot_dj(m), wx = cx + slot_di(m);
            const V3 xj = {sh.wx[0][wy][wx], sh.wx[1][wy][wx], sh.wx[2][wy][wx]};
            const V3 vj = {sh.wv[0][wy][wx], sh.wv[1][wy][wx], sh.wv[2][wy][wx]};
            V3 f;
            float K[6], P[6];
            spring_terms(xi, xj, vi, vj, in.L0, in.ks, in.kd, f, K, P);
#pragma unroll
            for (int q = 0; q < 6; q++) C[q] += h * (in.kd * P[q]) + hh * K[q];
            const V3 kw = symmv(K, V3{vi.x - vj.x, vi.y - vj.y, vi.z - vj.z});
            acc = {acc.x + f.x, acc.y + f.y, acc.z + f.z};
            kv = {kv.x + kw.x, kv.y + kw.y, kv.z + kw.z};
            if ((m >> 13) & 1u) {  // last spring of this pair
                if ((m >> 14) & 1u) {
                    const int plane = (m >> 9) & 15;
#pragma unroll
                    for (int q = 0; q < 6; q++)
                        sto(c.blocks + (size_t)q * N, (uint32_t)(plane * 6 * N + i), C[q]);
                }
                const V3 dvj = {sh.wdv[0][wy][wx], sh.wdv[1][wy][wx], sh.wdv[2][wy][wx]};
                V3 wd = {dvj.x - dvi.x, dvj.y - dvi.y, dvj.z - dvi.z};
                V3 a = symmv(C, wd);
                adv = {adv.x + a.x, adv.y + a.y, adv.z + a.z};
                dg = {dg.x - C[0], dg.y - C[1], dg.z - C[2]};
#pragma unroll
                for (int q = 0; q < 6; q++) C[q] = 0.0f;
            }
        }
        V3 b;
        b.x = pinned ? 0.0f : h * (acc.x + h * kv.x);
        b.y = pinned ? 0.0f : h * (acc.y + h * kv.y);
        b.z = pinned ? 0.0f : h * (acc.z + h * kv.z);
        st3o(c.b, N, i, b);
        V3 r = pinned ? V3{0.0f, 0.0f, 0.0f} : V3{b.x - adv.x, b.y - adv.y, b.z - adv.z};
        st3o(c.r, N, i, r);
        if (s.flags & OC_FLAG_JACOBI) {
            const V3 pv = {jacobi_inv(dg.x), jacobi_inv(dg.y), jacobi_inv(dg.z)};
            st3o(c.pinv, N, i, pv);
            const V3 z = {pv.x * r.x, pv.y * r.y, pv.z * r.z};
            st3o(c.s, N, i, z);
            st3o(c.d0, N, i, z);
            t = dot3(r, z);
        } else {
            st3o(c.d0, N, i, r);
            t = dot3(r, r);
        }
    }
    float p = tile_sum<NT>(t, sh.ws);
    if (threadIdx.x == 0) c.del_part[tile] = p;
}

// ---------------------------------------------------------------------------
// assembly, stencil assembly form: every spring evaluated once per tile
// ---------------------------------------------------------------------------
// A pair's owner is its lower-index vertex; the partner sits at one of six
// offsets (dx, dy) from it (owned direction o, owned_k).  The assembly visits
// the owned directions one after another.  In each, the block evaluates the
// springs owned by its tile's vertices and by the owners just outside the
// tile whose partner is inside (the direction's "strip"), once each, from
// the owner's side; the results (force, K (v_owner - v_partner) and the
// pair-block term) go to LDS.  Then every vertex adds, in its own stencil
// order, the pair it is partner of (the owner's results negated) and the
// pair it owns.  Negating the owner's force and K w equals evaluating from
// the partner's side (dp, f and K w change sign exactly, K and P are even in
// dp) up to the sign of zero, and these sums start at +0, where a signed
// zero cannot change a sum; so the results are the per-end kernel's bits.
// A second spring of a pair (the reference's duplicated last bends) is
// evaluated by each end itself.

template <int TX, int TY>
struct AssembleStShared {
    static constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    // columns 0 .. TX TY - 1: this direction's pairs owned in the tile;
    // then the strips of every direction, all evaluated before the first
    static constexpr int NR = TX * TY + strip_total<TX, TY>();
    float wx[3][WY][WX];
    float wv[3][WY][WX];
    float wdv[3][WY][WX];
    uint32_t wm[WY][WX];
    float res[12][NR];  // per evaluated pair: f, K w, block term
    float ws[TX * TY / 64];
    float bc;
};

// UPD as in k_assemble.
template <int TX, int TY, bool UPD>
__global__ __launch_bounds__(TX* TY, 4) void k_assemble_st(DevCloth c, StepScalars s) {
    constexpr int NT = TX * TY;
    using SH = AssembleStShared<TX, TY>;
    constexpr int WX = SH::WX, WY = SH::WY;
    constexpr int NWIN = (WX * WY + NT - 1) / NT;
    static_assert(strip_total<TX, TY>() <= NT, "the strips must fit one round of the block");
    __shared__ SH sh;
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int tile = tile_of_block(blockIdx.x, c.nt);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int N = c.N, nx = c.nx, i = gj * nx + gi;
    if (blockIdx.x == 0) begin_solve<UPD>(c, s, &sh.bc);
    auto own_cst = [&](int m, int o, int q, int g) {
        return ldo(c.cst, (uint32_t)(((m * kOwned + o) * 3 + q) * N + g));
    };
    // this thread's strip column (owner outside the tile, partner inside):
    // the strips of all directions are evaluated in one pass, packed into the
    // first waves, so no phase below waits on a wave with two evaluations
    int so = 0, swx = 0, swy = 0;
    bool sin = false;
    float sL0 = 0.0f, sks = 0.0f, skd = 0.0f;
    if ((int)threadIdx.x < strip_total<TX, TY>()) {
        int ss;
        strip_of_column<TX, TY>(threadIdx.x, so, ss);
        strip_owner<TX, TY>(so, ss, swx, swy);
        const int gx = bx * TX + swx, gy = by * TY + swy;
        if (gx >= 0 && gx < nx && gy >= 0 && gy < c.ny) {
            const int g = gy * nx + gx;
            sin = true;
            sL0 = own_cst(0, so, 0, g);
            sks = own_cst(0, so, 1, g);
            skd = own_cst(0, so, 2, g);
        }
    }
    // the window: x, v, dv and the stencil masks of the tile and its halo
    const int x0 = bx * TX - H, y0 = by * TY - H;
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        if (idx < WX * WY) {
            const int wx = idx % WX, wy = idx / WX;
            const int gx = x0 + wx, gy = y0 + wy;
            V3 xw = {0.0f, 0.0f, 0.0f}, vw = xw, dw = xw;
            uint32_t mw = 0;
            if (gx >= 0 && gx < nx && gy >= 0 && gy < c.ny) {
                const int g = gy * nx + gx;
                mw = ldo(c.asm_mask, (uint32_t)g);
                xw = ld3o(c.x, N, g);
                vw = ld3o(c.v, N, g);
                if (UPD) {
                    const V3 dp = ld3o(c.dv, N, g);
                    vw = {vw.x + dp.x, vw.y + dp.y, vw.z + dp.z};
                    xw = {xw.x + s.h * vw.x, xw.y + s.h * vw.y, xw.z + s.h * vw.z};
                    if ((s.flags & OC_FLAG_GROUND_CLAMP) && xw.y < 0.0f) xw.y = 0.0f;
                    dw = dp;
                } else if (s.warm) {
                    dw = ld3o(c.dv, N, g);
                }
            }
            sh.wx[0][wy][wx] = xw.x;
            sh.wx[1][wy][wx] = xw.y;
            sh.wx[2][wy][wx] = xw.z;
            sh.wv[0][wy][wx] = vw.x;
            sh.wv[1][wy][wx] = vw.y;
            sh.wv[2][wy][wx] = vw.z;
            sh.wdv[0][wy][wx] = dw.x;
            sh.wdv[1][wy][wx] = dw.y;
            sh.wdv[2][wy][wx] = dw.z;
            sh.wm[wy][wx] = mw;
        }
    }
    // the first direction's constants of this vertex's pair
    float oL0 = 0.0f, oks = 0.0f, okd = 0.0f;
    auto prefetch = [&](int o) {
        if (own) {
            oL0 = own_cst(0, o, 0, i);
            oks = own_cst(0, o, 1, i);
            okd = own_cst(0, o, 2, i);
        }
    };
    prefetch(0);
    __syncthreads();

    const float h = s.h, hh = s.hh;
    const int cx = lx + H, cy = ly + H;
    const V3 xi = {sh.wx[0][cy][cx], sh.wx[1][cy][cx], sh.wx[2][cy][cx]};
    const V3 vi = {sh.wv[0][cy][cx], sh.wv[1][cy][cx], sh.wv[2][cy][cx]};
    const V3 dvi = {sh.wdv[0][cy][cx], sh.wdv[1][cy][cx], sh.wdv[2][cy][cx]};
    const uint32_t mi = own ? sh.wm[cy][cx] : 0u;
    bool pinned = true;
    V3 acc = {0.0f, 0.0f, 0.0f}, kv = {0.0f, 0.0f, 0.0f};
    V3 adv = {0.0f, 0.0f, 0.0f}, dg = {0.0f, 0.0f, 0.0f};
    if (own) {
        pinned = ldo(c.pin, (uint32_t)i) != 0;
        if (!s.warm) st3o(c.dv, N, i, dvi);
        if (UPD) {
            st3o(c.xo, N, i, xi);
            st3o(c.vo, N, i, vi);
            if (!(isfinite(xi.x) && isfinite(xi.y) && isfinite(xi.z) && isfinite(vi.x) &&
                  isfinite(vi.y) && isfinite(vi.z)))
                atomicOr(c.ctl + 3, OC_SOLVE_NONFINITE);
        }
        if (!pinned) acc = {0.0f + s.mass * s.gx, 0.0f + s.mass * s.gy, 0.0f + s.mass * s.gz};
        if (!pinned && s.damp != 0.0f)
            acc = {acc.x + s.damp * vi.x, acc.y + s.damp * vi.y, acc.z + s.damp * vi.z};
        adv = {s.md * dvi.x, s.md * dvi.y, s.md * dvi.z};
        dg = {s.md, s.md, s.md};
    }
    float C[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    auto window3 = [&](float (&w)[3][WY][WX], int px, int py) {
        return V3{w[0][py][px], w[1][py][px], w[2][py][px]};
    };
    // Add one spring's terms (from this vertex's side) to the pair's sums.
    auto add_spring = [&](const SpringOut& r) {
#pragma unroll
        for (int q = 0; q < 6; q++) C[q] += r.c[q];
        acc = {acc.x + r.f.x, acc.y + r.f.y, acc.z + r.f.z};
        kv = {kv.x + r.kw.x, kv.y + r.kw.y, kv.z + r.kw.z};
    };
    // The second spring of the pair with the neighbour at window (px, py),
    // from this vertex's side (constants of the owner g at multiplicity 1).
    auto add_second = [&](int o, int g, int px, int py) {
        const SpringOut r = eval_spring(xi, window3(sh.wx, px, py), vi, window3(sh.wv, px, py),
                                        own_cst(1, o, 0, g), own_cst(1, o, 1, g), own_cst(1, o, 2, g),
                                        h, hh);
        add_spring(r);
    };
    // The pair is complete: its block (when owned), A dv and diag(A) terms.
    auto finish_pair = [&](int px, int py, int k_store) {
        if (k_store >= 0) {
            const int plane = c.stencil_plane[k_store];
#pragma unroll
            for (int q = 0; q < 6; q++)
                sto(c.blocks + (size_t)q * N, (uint32_t)(plane * 6 * N + i), C[q]);
        }
        const V3 dvj = window3(sh.wdv, px, py);
        const V3 a = symmv(C, V3{dvj.x - dvi.x, dvj.y - dvi.y, dvj.z - dvi.z});
        adv = {adv.x + a.x, adv.y + a.y, adv.z + a.z};
        dg = {dg.x - C[0], dg.y - C[1], dg.z - C[2]};
#pragma unroll
        for (int q = 0; q < 6; q++) C[q] = 0.0f;
    };

    // The result stored at LDS column r (the owner's side).
    auto stored = [&](int r) {
        SpringOut e;
        e.f = {sh.res[0][r], sh.res[1][r], sh.res[2][r]};
        e.kw = {sh.res[3][r], sh.res[4][r], sh.res[5][r]};
#pragma unroll
        for (int q = 0; q < 6; q++) e.c[q] = sh.res[6 + q][r];
        return e;
    };
    // ---- the strips: column NT + t holds strip column t's pair (the owner's side)
    if (sin && ((sh.wm[swy + H][swx + H] >> owned_k(so)) & 1u)) {
        const int px = swx + H, py = swy + H, dx = own_dx(so), dy = own_dy(so);
        const SpringOut e = eval_spring(window3(sh.wx, px, py), window3(sh.wx, px + dx, py + dy),
                                        window3(sh.wv, px, py), window3(sh.wv, px + dx, py + dy),
                                        sL0, sks, skd, h, hh);
        const int r = NT + threadIdx.x;
        sh.res[0][r] = e.f.x;
        sh.res[1][r] = e.f.y;
        sh.res[2][r] = e.f.z;
        sh.res[3][r] = e.kw.x;
        sh.res[4][r] = e.kw.y;
        sh.res[5][r] = e.kw.z;
#pragma unroll
        for (int q = 0; q < 6; q++) sh.res[6 + q][r] = e.c[q];
    }
    SpringOut held{};  // this vertex's k = 7 pair, added after k = 5 and k = 6
#pragma unroll 1
    for (int o = 0; o < kOwned; o++) {
        const int dx = own_dx(o), dy = own_dy(o);
        const int ko = owned_k(o), kp = owned_partner_k(o);
        // ---- evaluate this vertex's pair in direction o
        if (own && ((mi >> ko) & 1u)) {
            const SpringOut e = eval_spring(xi, window3(sh.wx, cx + dx, cy + dy), vi,
                                            window3(sh.wv, cx + dx, cy + dy), oL0, oks, okd, h, hh);
            const int r = threadIdx.x;
            sh.res[0][r] = e.f.x;
            sh.res[1][r] = e.f.y;
            sh.res[2][r] = e.f.z;
            sh.res[3][r] = e.kw.x;
            sh.res[4][r] = e.kw.y;
            sh.res[5][r] = e.kw.z;
#pragma unroll
            for (int q = 0; q < 6; q++) sh.res[6 + q][r] = e.c[q];
        }
        if (o + 1 < kOwned) prefetch(o + 1);
        __syncthreads();
        // ---- accumulate, in this vertex's stencil order
        if (own && ((mi >> kp) & 1u)) {  // partner of the pair owned at -(dx, dy)
            const int wx = lx - dx, wy = ly - dy;
            const int r = (wx >= 0 && wx < TX && wy >= 0 && wy < TY)
                              ? wy * TX + wx
                              : NT + strip_base<TX, TY>(o) + strip_index<TX, TY>(o, wx, wy);
            SpringOut e = stored(r);
            e.f = {0.0f - e.f.x, 0.0f - e.f.y, 0.0f - e.f.z};
            e.kw = {0.0f - e.kw.x, 0.0f - e.kw.y, 0.0f - e.kw.z};
            add_spring(e);
            if ((mi >> (16 + kp)) & 1u) add_second(o, i - dy * nx - dx, cx - dx, cy - dy);
            finish_pair(cx - dx, cy - dy, -1);
        }
        if (o == 2) {
            if (own && ((mi >> ko) & 1u)) held = stored(threadIdx.x);  // k = 7 follows k = 5, 6
        } else if (own) {
#pragma unroll
            for (int t = 0; t < 2; t++) {  // k = 6, then the held k = 7; else just ko
                const int oo = o == 3 ? (t == 0 ? 3 : 2) : o;
                if (t == 1 && o != 3) break;
                const int kk = owned_k(oo), ddx = own_dx(oo), ddy = own_dy(oo);
                if (!((mi >> kk) & 1u)) continue;
                add_spring(t == 0 ? stored(threadIdx.x) : held);
                if ((mi >> (16 + kk)) & 1u) add_second(oo, i, cx + ddx, cy + ddy);
                finish_pair(cx + ddx, cy + ddy, kk);
            }
        }
        __syncthreads();
    }

    float t = 0.0f;
    if (own) {
        V3 b;
        b.x = pinned ? 0.0f : h * (acc.x + h * kv.x);
        b.y = pinned ? 0.0f : h * (acc.y + h * kv.y);
        b.z = pinned ? 0.0f : h * (acc.z + h * kv.z);
        st3o(c.b, N, i, b);
        V3 r = pinned ? V3{0.0f, 0.0f, 0.0f} : V3{b.x - adv.x, b.y - adv.y, b.z - adv.z};
        st3o(c.r, N, i, r);
        if (s.flags & OC_FLAG_JACOBI) {
            const V3 pv = {jacobi_inv(dg.x), jacobi_inv(dg.y), jacobi_inv(dg.z)};
            st3o(c.pinv, N, i, pv);
            const V3 z = {pv.x * r.x, pv.y * r.y, pv.z * r.z};
            st3o(c.s, N, i, z);
            st3o(c.d0, N, i, z);
            t = dot3(r, z);
        } else {
            st3o(c.d0, N, i, r);
            t = dot3(r, r);
        }
    }
    float p = tile_sum<NT>(t, sh.ws);
    if (threadIdx.x == 0) c.del_part[tile] = p;
}

// The assembly of a cloth of few tiles: blocks of TX x TY vertices, rows of
// the reduction's tiles; each wave's sum of r.z goes to c.row_part (tile, row
// of the tile).  A few tiles leave most CUs idle, and what takes the time is
// a wave's own chain (about 9.5 cycles per instruction with one or two waves
// on a SIMD: 2000 per direction to evaluate, 2500 to accumulate).  So a block
// is half a tile, the six directions go in three pairs whose evaluations have
// no branch and overlap, what an accumulation reads is read before it starts,
// and second springs are evaluated ahead: 21x21 20.5 -> 17.0 us, 90x71
// 21.9 -> 16.9, 128x128 21.6 -> 16.9 (half tiles alone, direction by
// direction, 24, 22.5 and 21.4).
template <int TX, int TY>
struct AssemblePairShared {
    static constexpr int WX = TX + 2 * H, WY = TY + 2 * H, NT = TX * TY, NS = strip_total<TX, TY>();
    float wx[3][WY][WX];
    float wv[3][WY][WX];
    float wdv[3][WY][WX];
    uint32_t wm[WY][WX];
    float res[2][12 * NT];  // per direction of the pair 12 planes: f, K w, block term
    float second[2][12 * NT];
    float strip[12 * NS];
    float bc;
};

template <int TX, int TY, bool UPD>
__global__ __launch_bounds__(TX* TY, 2) void k_assemble_pairs(DevCloth c, StepScalars s) {
    constexpr int NT = TX * TY;
    using SH = AssemblePairShared<TX, TY>;
    constexpr int WX = SH::WX, WY = SH::WY, NS = SH::NS;
    constexpr int NWIN = (WX * WY + NT - 1) / NT;
    constexpr int NSR = (NS + NT - 1) / NT;  // rounds of the strips
    __shared__ SH sh;
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int tile = tile_of_block(blockIdx.x, gridDim.x);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int N = c.N, nx = c.nx, i = gj * nx + gi;
    if (blockIdx.x == 0) begin_solve<UPD>(c, s, &sh.bc);
    auto own_cst = [&](int m, int o, int q, int g) {
        return ldo(c.cst, (uint32_t)(((m * kOwned + o) * 3 + q) * N + g));
    };
    const uint32_t mi = own ? ldo(c.asm_mask, (uint32_t)i) : 0u;
    float L0[2], ks[2], kd[2];  // of the pair of directions to come
    auto prefetch = [&](int p) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int g = own ? i : 0;
            L0[q] = own_cst(0, 2 * p + q, 0, g);
            ks[q] = own_cst(0, 2 * p + q, 1, g);
            kd[q] = own_cst(0, 2 * p + q, 2, g);
        }
    };
    prefetch(0);
    // this thread's strip springs (owner outside the block, partner inside)
    int so[NSR], swx[NSR], swy[NSR];
    bool sin[NSR];
    float sL0[NSR], sks[NSR], skd[NSR];
#pragma unroll
    for (int n = 0; n < NSR; n++) {
        so[n] = swx[n] = swy[n] = 0;
        sin[n] = false;
        sL0[n] = sks[n] = skd[n] = 0.0f;
        const int col = threadIdx.x + n * NT;
        if (col < NS) {
            int ss;
            strip_of_column<TX, TY>(col, so[n], ss);
            strip_owner<TX, TY>(so[n], ss, swx[n], swy[n]);
            const int gx = bx * TX + swx[n], gy = by * TY + swy[n];
            if (gx >= 0 && gx < nx && gy >= 0 && gy < c.ny) {
                const int g = gy * nx + gx;
                sin[n] = true;
                sL0[n] = own_cst(0, so[n], 0, g);
                sks[n] = own_cst(0, so[n], 1, g);
                skd[n] = own_cst(0, so[n], 2, g);
            }
        }
    }
    // the window: x, v, dv and the stencil masks of the tile and its halo
    const int x0 = bx * TX - H, y0 = by * TY - H;
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        if (idx < WX * WY) {
            const int wx = idx % WX, wy = idx / WX;
            const int gx = x0 + wx, gy = y0 + wy;
            V3 xw = {0.0f, 0.0f, 0.0f}, vw = xw, dw = xw;
            uint32_t mw = 0;
            if (gx >= 0 && gx < nx && gy >= 0 && gy < c.ny) {
                const int g = gy * nx + gx;
                mw = ldo(c.asm_mask, (uint32_t)g);
                xw = ld3o(c.x, N, g);
                vw = ld3o(c.v, N, g);
                if (UPD) {
                    const V3 dp = ld3o(c.dv, N, g);
                    vw = {vw.x + dp.x, vw.y + dp.y, vw.z + dp.z};
                    xw = {xw.x + s.h * vw.x, xw.y + s.h * vw.y, xw.z + s.h * vw.z};
                    if ((s.flags & OC_FLAG_GROUND_CLAMP) && xw.y < 0.0f) xw.y = 0.0f;
                    dw = dp;
                } else if (s.warm) {
                    dw = ld3o(c.dv, N, g);
                }
            }
            sh.wx[0][wy][wx] = xw.x;
            sh.wx[1][wy][wx] = xw.y;
            sh.wx[2][wy][wx] = xw.z;
            sh.wv[0][wy][wx] = vw.x;
            sh.wv[1][wy][wx] = vw.y;
            sh.wv[2][wy][wx] = vw.z;
            sh.wdv[0][wy][wx] = dw.x;
            sh.wdv[1][wy][wx] = dw.y;
            sh.wdv[2][wy][wx] = dw.z;
            sh.wm[wy][wx] = mw;
        }
    }
    // the first two second springs of this vertex's pairs, in stencil order
    float eL0[2] = {0.0f, 0.0f}, eks[2] = {0.0f, 0.0f}, ekd[2] = {0.0f, 0.0f};
    int ek[2] = {-1, -1};
    {
        uint32_t m = mi >> 16;
#pragma unroll
        for (int q = 0; q < 2; q++)
            if (m) {
                const int k = __ffs(m) - 1, o = owned_index(k);
                const int g = stencil_owner(k) ? i : i + stencil_dj(k) * nx + stencil_di(k);
                ek[q] = k;
                eL0[q] = own_cst(1, o, 0, g);
                eks[q] = own_cst(1, o, 1, g);
                ekd[q] = own_cst(1, o, 2, g);
                m &= m - 1u;
            }
    }
    __syncthreads();

    const float h = s.h, hh = s.hh;
    const int cx = lx + H, cy = ly + H;
    const V3 xi = {sh.wx[0][cy][cx], sh.wx[1][cy][cx], sh.wx[2][cy][cx]};
    const V3 vi = {sh.wv[0][cy][cx], sh.wv[1][cy][cx], sh.wv[2][cy][cx]};
    const V3 dvi = {sh.wdv[0][cy][cx], sh.wdv[1][cy][cx], sh.wdv[2][cy][cx]};
    bool pinned = true;
    V3 acc = {0.0f, 0.0f, 0.0f}, kv = {0.0f, 0.0f, 0.0f};
    V3 adv = {0.0f, 0.0f, 0.0f}, dg = {0.0f, 0.0f, 0.0f};
    if (own) {
        pinned = ldo(c.pin, (uint32_t)i) != 0;
        if (!s.warm) st3o(c.dv, N, i, dvi);
        if (UPD) {
            st3o(c.xo, N, i, xi);
            st3o(c.vo, N, i, vi);
            if (!(isfinite(xi.x) && isfinite(xi.y) && isfinite(xi.z) && isfinite(vi.x) &&
                  isfinite(vi.y) && isfinite(vi.z)))
                atomicOr(c.ctl + 3, OC_SOLVE_NONFINITE);
        }
        if (!pinned) acc = {0.0f + s.mass * s.gx, 0.0f + s.mass * s.gy, 0.0f + s.mass * s.gz};
        if (!pinned && s.damp != 0.0f)
            acc = {acc.x + s.damp * vi.x, acc.y + s.damp * vi.y, acc.z + s.damp * vi.z};
        adv = {s.md * dvi.x, s.md * dvi.y, s.md * dvi.z};
        dg = {s.md, s.md, s.md};
    }
    auto window3 = [&](float (&w)[3][WY][WX], int px, int py) {
        return V3{w[0][py][px], w[1][py][px], w[2][py][px]};
    };
    auto put = [&](float* p, int stride, const SpringOut& e) {
        p[0] = e.f.x;
        p[stride] = e.f.y;
        p[2 * stride] = e.f.z;
        p[3 * stride] = e.kw.x;
        p[4 * stride] = e.kw.y;
        p[5 * stride] = e.kw.z;
#pragma unroll
        for (int q = 0; q < 6; q++) p[(6 + q) * stride] = e.c[q];
    };
    auto get = [&](const float* p, int stride) {
        SpringOut e;
        e.f = {p[0], p[stride], p[2 * stride]};
        e.kw = {p[3 * stride], p[4 * stride], p[5 * stride]};
#pragma unroll
        for (int q = 0; q < 6; q++) e.c[q] = p[(6 + q) * stride];
        return e;
    };
    // ---- the strips' springs, and this vertex's second springs
#pragma unroll 1
    for (int n = 0; n < NSR + 2; n++) {
        int ax = cx, ay = cy, px = cx, py = cy, stride = NT;
        float l0 = 0.0f, k0 = 0.0f, d0 = 0.0f;
        float* dst = nullptr;
#pragma unroll
        for (int q = 0; q < NSR; q++)
            if (n == q && sin[q] && ((sh.wm[swy[q] + H][swx[q] + H] >> owned_k(so[q])) & 1u)) {
                ax = swx[q] + H;
                ay = swy[q] + H;
                px = ax + own_dx(so[q]);
                py = ay + own_dy(so[q]);
                l0 = sL0[q];
                k0 = sks[q];
                d0 = skd[q];
                dst = sh.strip + threadIdx.x + q * NT;
                stride = NS;
            }
#pragma unroll
        for (int q = 0; q < 2; q++)
            if (n == NSR + q && ek[q] >= 0) {
                px = cx + stencil_di(ek[q]);
                py = cy + stencil_dj(ek[q]);
                l0 = eL0[q];
                k0 = eks[q];
                d0 = ekd[q];
                dst = sh.second[q] + threadIdx.x;
            }
        if (dst)
            put(dst, stride,
                eval_spring(window3(sh.wx, ax, ay), window3(sh.wx, px, py), window3(sh.wv, ax, ay), window3(sh.wv, px, py),
                            l0, k0, d0, h, hh));
    }
    // One pair of this vertex: position k, its spring's terms from this side,
    // the neighbour's dv.
    auto add_pair = [&](int k, const SpringOut& r, V3 dvj, bool owner) {
        if (!((mi >> k) & 1u)) return;
        float C[6];
        auto add = [&](const SpringOut& e) {
#pragma unroll
            for (int q = 0; q < 6; q++) C[q] += e.c[q];
            acc = {acc.x + e.f.x, acc.y + e.f.y, acc.z + e.f.z};
            kv = {kv.x + e.kw.x, kv.y + e.kw.y, kv.z + e.kw.z};
        };
#pragma unroll
        for (int q = 0; q < 6; q++) C[q] = 0.0f;
        add(r);
        if ((mi >> (16 + k)) & 1u) {
            if (k == ek[0] || k == ek[1]) {
                add(get(sh.second[k == ek[0] ? 0 : 1] + threadIdx.x, NT));
            } else {  // a third one (no topology of the reference's)
                const int o = owned_index(k), di = stencil_di(k), dj = stencil_dj(k), g = owner ? i : i + dj * nx + di;
                add(eval_spring(xi, window3(sh.wx, cx + di, cy + dj), vi, window3(sh.wv, cx + di, cy + dj),
                                own_cst(1, o, 0, g), own_cst(1, o, 1, g), own_cst(1, o, 2, g), h, hh));
            }
        }
        if (owner) {
            const int plane = c.stencil_plane[k];
#pragma unroll
            for (int q = 0; q < 6; q++) sto(c.blocks + (size_t)q * N, (uint32_t)(plane * 6 * N + i), C[q]);
        }
        const V3 a = symmv(C, V3{dvj.x - dvi.x, dvj.y - dvi.y, dvj.z - dvi.z});
        adv = {adv.x + a.x, adv.y + a.y, adv.z + a.z};
        dg = {dg.x - C[0], dg.y - C[1], dg.z - C[2]};
    };
#pragma unroll 1
    for (int p = 0; p < kOwned / 2; p++) {
        const int oa = 2 * p, ob = 2 * p + 1;
        const int ax = own_dx(oa), ay = own_dy(oa), bx2 = own_dx(ob), by2 = own_dy(ob);
        // ---- evaluate this vertex's pairs in both directions (past the
        // cloth's edge: of the window's zeros, not used)
        const SpringOut ea = eval_spring(xi, window3(sh.wx, cx + ax, cy + ay), vi, window3(sh.wv, cx + ax, cy + ay), L0[0],
                                         ks[0], kd[0], h, hh);
        const SpringOut eb = eval_spring(xi, window3(sh.wx, cx + bx2, cy + by2), vi, window3(sh.wv, cx + bx2, cy + by2),
                                         L0[1], ks[1], kd[1], h, hh);
        put(sh.res[0] + threadIdx.x, NT, ea);
        put(sh.res[1] + threadIdx.x, NT, eb);
        if (p + 1 < kOwned / 2) prefetch(p + 1);
        __syncthreads();
        // ---- accumulate, in this vertex's stencil order
        auto partner = [&](int q, int o, int dx, int dy) {
            const int wx = lx - dx, wy = ly - dy;
            const bool in = wx >= 0 && wx < TX && wy >= 0;
            const bool have = (mi >> owned_partner_k(o)) & 1u;
            const float* src = sh.res[q] + (in ? wy * TX + wx : 0);
            int stride = NT;
            if (!in && have) {
                src = sh.strip + strip_base<TX, TY>(o) + strip_index<TX, TY>(o, wx, wy);
                stride = NS;
            }
            SpringOut e = get(src, stride);
            e.f = {0.0f - e.f.x, 0.0f - e.f.y, 0.0f - e.f.z};
            e.kw = {0.0f - e.kw.x, 0.0f - e.kw.y, 0.0f - e.kw.z};
            return e;
        };
        const SpringOut pa = partner(0, oa, ax, ay), pb = partner(1, ob, bx2, by2);
        const V3 va = window3(sh.wdv, cx - ax, cy - ay), vb = window3(sh.wdv, cx - bx2, cy - by2);
        const V3 ua = window3(sh.wdv, cx + ax, cy + ay), ub = window3(sh.wdv, cx + bx2, cy + by2);
        add_pair(owned_partner_k(oa), pa, va, false);
        if (p == 1) {  // 4, 5, 6, 7: the diagonals
            add_pair(owned_partner_k(ob), pb, vb, false);
            add_pair(owned_k(ob), eb, ub, true);
            add_pair(owned_k(oa), ea, ua, true);
        } else {
            add_pair(owned_k(oa), ea, ua, true);
            add_pair(owned_partner_k(ob), pb, vb, false);
            add_pair(owned_k(ob), eb, ub, true);
        }
        __syncthreads();
    }

    float t = 0.0f;
    if (own) {
        V3 b;
        b.x = pinned ? 0.0f : h * (acc.x + h * kv.x);
        b.y = pinned ? 0.0f : h * (acc.y + h * kv.y);
        b.z = pinned ? 0.0f : h * (acc.z + h * kv.z);
        st3o(c.b, N, i, b);
        V3 r = pinned ? V3{0.0f, 0.0f, 0.0f} : V3{b.x - adv.x, b.y - adv.y, b.z - adv.z};
        st3o(c.r, N, i, r);
        if (s.flags & OC_FLAG_JACOBI) {
            const V3 pv = {jacobi_inv(dg.x), jacobi_inv(dg.y), jacobi_inv(dg.z)};
            st3o(c.pinv, N, i, pv);
            const V3 z = {pv.x * r.x, pv.y * r.y, pv.z * r.z};
            st3o(c.s, N, i, z);
            st3o(c.d0, N, i, z);
            t = dot3(r, z);
        } else {
            st3o(c.d0, N, i, r);
            t = dot3(r, r);
        }
    }
    const float w = wave_sum(t);
    if (lx == 0) c.row_part[(gj / kTileY * c.ntx + bx) * kTileY + gj % kTileY] = w;
}

// ---------------------------------------------------------------------------
// CG iteration k, part 1: direction update on the tile + halo, q = S A d
// ---------------------------------------------------------------------------
template <int TX, int TY>
struct SpmvShared {
    static constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    float wd[3][WY][WX];
    float ws[TX * TY / 64];
    float bc;
};

// One block's share of CG iteration k, part 1.  read_done: take the stop
// flag of earlier launches from c.ctl[0] (multi-kernel form).  Returns true
// when the solve has stopped (every block decides alike).  STENCIL: the
// cloth's pairs follow the kStencil order (c.stencil), so a 12-bit mask per
// vertex replaces the WP slot metas and every slot's offset, owner and plane
// are constants; the sums run in the same pair order either way.
// LEAN (stencil form): the blocks are read as they are used instead of up
// front, for a kernel whose registers the hoisted form would spill.
template <int TX, int TY, int WP, bool STENCIL = false, bool LEAN = false>
__device__ inline bool spmv_phase(const DevCloth& c, const StepScalars& s, int k, bool read_done,
                                  SpmvShared<TX, TY>& sh, int vb) {
    constexpr int NT = TX * TY;
    constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    constexpr int NWIN = (WX * WY + NT - 1) / NT;
    const int nt = c.nt, N = c.N;
    const int tile = tile_of_block(vb, nt);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int i = gj * c.nx + gi;

    // ---- loads that do not depend on beta (the stencil mask first: the
    // block loads wait for it)
    uint32_t mask = 0;
    if constexpr (STENCIL) mask = own ? ldo(c.pair_mask, (uint32_t)i) : 0u;
    const int done = read_done ? c.ctl[0] : 0;
    const float delta0 = c.scal[0];
    const float delta_old = k > 0 ? c.scal[k - 1] : 0.0f;
    float pv[kPartialRegs];
    if (threadIdx.x < 64) partial_load(c.del_part + (size_t)k * nt, nt, pv);
    const float* dprev = (k & 1) ? c.d0 : c.d1;
    float* dcur = (k & 1) ? c.d1 : c.d0;
    const float* zsrc = (s.flags & OC_FLAG_JACOBI) ? c.s : c.r;  // d = z + beta d
    const int x0 = bx * TX - H, y0 = by * TY - H;
    V3 wr[NWIN], wp[NWIN];
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        const int gx = x0 + idx % WX, gy = y0 + idx / WX;
        wr[n] = wp[n] = V3{0.0f, 0.0f, 0.0f};
        if (idx < WX * WY && gx >= 0 && gx < c.nx && gy >= 0 && gy < c.ny) {
            const int g = gy * c.nx + gx;
            if (k == 0) {
                wr[n] = ld3o(c.d0, N, g);
            } else {
                wr[n] = ld3o(zsrc, N, g);
                wp[n] = ld3o(dprev, N, g);
            }
        }
    }
    constexpr int NS = LEAN ? 1 : STENCIL ? kStencil : WP;
    uint16_t m[NS];
    float C[NS][6];
    auto stencil_block = [&](int k, float (&b)[6]) {
        const int di = stencil_di(k), dj = stencil_dj(k);
        const uint32_t blk = stencil_owner(k) ? (uint32_t)i : (uint32_t)(i + dj * c.nx + di);
        const uint32_t off = blk + (uint32_t)c.stencil_plane[k] * 6u * (uint32_t)N;
        if ((mask >> k) & 1u) {
#pragma unroll
            for (int q = 0; q < 6; q++) b[q] = ldo(c.blocks, off + (uint32_t)(q * N));
        } else {
#pragma unroll
            for (int q = 0; q < 6; q++) b[q] = 0.0f;
        }
    };
    if constexpr (STENCIL && !LEAN) {
#pragma unroll
        for (int k = 0; k < kStencil; k++) stencil_block(k, C[k]);
    } else if constexpr (!STENCIL) {
#pragma unroll
        for (int sl = 0; sl < WP; sl++) {
            m[sl] = (own && sl < c.wp) ? ldo(c.pair_m, (uint32_t)(sl * N + i)) : kEmptySlot;
            if (m[sl] != kEmptySlot) {
                const int j = i + slot_dj(m[sl]) * c.nx + slot_di(m[sl]);
                const int blk = ((m[sl] >> 12) & 1) ? i : j;
                const uint32_t b0 = (uint32_t)((m[sl] >> 8) & 15) * 6u * (uint32_t)N + (uint32_t)blk;
#pragma unroll
                for (int q = 0; q < 6; q++) C[sl][q] = ldo(c.blocks + (size_t)q * N, b0);
            } else {
#pragma unroll
                for (int q = 0; q < 6; q++) C[sl][q] = 0.0f;
            }
        }
    }
    const bool pinned = own ? ldo(c.pin, (uint32_t)i) != 0 : true;

    // ---- r.r of this iteration, stopping test, beta
    if (threadIdx.x < 64) {
        const float sum = partial_finish(c.del_part + (size_t)k * nt, nt, pv);
        if (threadIdx.x == 0) sh.bc = sum;
    }
    __syncthreads();
    if (done) return true;
    const float delta = sh.bc;
    const float thresh = s.tol_mode == 1 ? s.tol2 * (k == 0 ? delta : delta0) : s.tol2;
    const bool stop = s.tol_mode != 2 && !(delta > thresh);
    if (vb == 0 && threadIdx.x == 0) {
        c.scal[k] = delta;
        if (stop) {
            c.ctl[0] = 1;
            c.ctl[1] = k;
        }
    }
    if (stop) return true;
    // beta = 0 once r.r has underflowed to 0 (fixed iteration counts)
    const float beta = (k > 0 && delta_old != 0.0f) ? delta / delta_old : 0.0f;

    // ---- d = r + beta d on tile + halo into LDS; the tile's own d to memory
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        if (idx < WX * WY) {
            const int wx = idx % WX, wy = idx / WX;
            V3 d = wr[n];
            if (k > 0) {
                d = {wr[n].x + beta * wp[n].x, wr[n].y + beta * wp[n].y, wr[n].z + beta * wp[n].z};
                const int gx = x0 + wx, gy = y0 + wy;
                if (wx >= H && wx < H + TX && wy >= H && wy < H + TY && gx < c.nx && gy < c.ny)
                    st3o(dcur, N, gy * c.nx + gx, d);
            }
            sh.wd[0][wy][wx] = d.x;
            sh.wd[1][wy][wx] = d.y;
            sh.wd[2][wy][wx] = d.z;
        }
    }
    __syncthreads();

    // ---- q = S A d
    float t = 0.0f;
    if (own) {
        const V3 di = {sh.wd[0][ly + H][lx + H], sh.wd[1][ly + H][lx + H], sh.wd[2][ly + H][lx + H]};
        V3 acc = {s.md * di.x, s.md * di.y, s.md * di.z};
        if constexpr (STENCIL) {
#pragma unroll
            for (int k = 0; k < kStencil; k++) {
                if (!((mask >> k) & 1u)) continue;
                const int wy = ly + H + stencil_dj(k), wx = lx + H + stencil_di(k);
                V3 w = {sh.wd[0][wy][wx] - di.x, sh.wd[1][wy][wx] - di.y, sh.wd[2][wy][wx] - di.z};
                if constexpr (LEAN) stencil_block(k, C[0]);
                V3 a = symmv(C[LEAN ? 0 : k], w);
                acc = {acc.x + a.x, acc.y + a.y, acc.z + a.z};
            }
        } else {
#pragma unroll
            for (int sl = 0; sl < WP; sl++) {
                if (m[sl] == kEmptySlot) break;
                const int wy = ly + H + slot_dj(m[sl]), wx = lx + H + slot_di(m[sl]);
                V3 w = {sh.wd[0][wy][wx] - di.x, sh.wd[1][wy][wx] - di.y, sh.wd[2][wy][wx] - di.z};
                V3 a = symmv(C[sl], w);
                acc = {acc.x + a.x, acc.y + a.y, acc.z + a.z};
            }
        }
        V3 q = pinned ? V3{0.0f, 0.0f, 0.0f} : acc;
        st3o(c.q, N, i, q);
        t = dot3(di, q);
    }
    float p = tile_sum<NT>(t, sh.ws);
    if (threadIdx.x == 0) c.sig_part[(size_t)k * nt + tile] = p;
    return false;
}

template <int TX, int TY, int WP, bool STENCIL>
__global__ __launch_bounds__(TX* TY) void k_cg_spmv(DevCloth c, StepScalars s, int k) {
    __shared__ SpmvShared<TX, TY> sh;
    spmv_phase<TX, TY, WP, STENCIL>(c, s, k, true, sh, blockIdx.x);
}

// ---------------------------------------------------------------------------
// single-reduction CG (OC_FLAG_CG_SINGLE_REDUCTION): one launch per iteration
// ---------------------------------------------------------------------------
// The Chronopoulos-Gear recurrence (s = 1): with u = P^-1 r and w = S A u the
// two dots gamma = r.u and delta = w.u of an iteration come from the same
// launch, so each iteration needs one reduction point, and one launch:
//   beta = gamma_k / gamma_{k-1},  alpha = gamma_k / (delta_k - beta gamma_k / alpha_{k-1})
//   p = u + beta p,  s = w + beta s  (s = S A p),  dv += alpha p,  r -= alpha s,
//   u = P^-1 r,  w = S A u,  partials of r.u and w.u.
// r, s and w are read on the tile's halo by neighbouring blocks while the
// launch writes their next values, so each has two buffers used by iteration
// parity; p and dv are only read on the tile itself.  The start (w0 = S A u0,
// delta_0) is the first launch of the standard SpMV, whose q is w0.  The
// arithmetic and guards are the oracle's cg_core_cg1, step for step.
template <int TX, int TY>
struct Cg1Shared {
    static constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    float wu[3][WY][WX];  // u_{k+1} on the tile and halo
    float rt[3][TY][TX];  // r_{k+1} of the tile
    float ws[TX * TY / 64];
    float ws2[TX * TY / 64];
    float bc, bc2;
};

// Buffers of iteration k: r_k, w_k, s_{k-1} are read, r_{k+1}, w_{k+1}, s_k
// written (parity k & 1).
struct Cg1Bufs {
    const float* r_in;
    float* r_out;
    const float* w_in;
    float* w_out;
    const float* s_in;
    float* s_out;
};
__device__ inline Cg1Bufs cg1_bufs(const DevCloth& c, int k) {
    Cg1Bufs b;
    const bool odd = (k & 1) != 0;
    b.r_in = odd ? c.r2 : c.r;
    b.r_out = odd ? c.r : c.r2;
    b.w_in = odd ? c.q2 : c.q;
    b.w_out = odd ? c.q : c.q2;
    b.s_in = odd ? c.s1 : c.s2;
    b.s_out = odd ? c.s2 : c.s1;
    return b;
}

template <int TX, int TY, int WP, bool STENCIL>
__global__ __launch_bounds__(TX* TY) void k_cg1(DevCloth c, StepScalars s, int k) {
    constexpr int NT = TX * TY;
    constexpr int WX = TX + 2 * H, WY = TY + 2 * H;
    constexpr int NWIN = (WX * WY + NT - 1) / NT;
    constexpr int NP = 8;  // partials per lane loaded up front, per dot
    __shared__ Cg1Shared<TX, TY> sh;
    const int nt = c.nt, N = c.N;
    const int tile = tile_of_block(blockIdx.x, nt);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int i = gj * c.nx + gi;
    const bool jac = (s.flags & OC_FLAG_JACOBI) != 0;
    const Cg1Bufs bf = cg1_bufs(c, k);

    // ---- loads that do not depend on the reduction
    const int done = c.ctl[0];
    const float gamma_old = k > 0 ? c.scal[k - 1] : 0.0f;
    const float alpha_old = k > 0 ? c.scal[c.cg1_alpha + k - 1] : 0.0f;
    const float gamma0 = c.scal[0];
    float pg[NP], pd[NP];
    if (threadIdx.x < 64) {
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int t = threadIdx.x + 64 * j;
            pg[j] = t < nt ? c.del_part[(size_t)k * nt + t] : 0.0f;
            pd[j] = t < nt ? c.sig_part[(size_t)k * nt + t] : 0.0f;
        }
    }
    const int x0 = bx * TX - H, y0 = by * TY - H;
    V3 wr[NWIN], ww[NWIN], wsv[NWIN], wpv[NWIN];
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        const int gx = x0 + idx % WX, gy = y0 + idx / WX;
        wr[n] = ww[n] = wsv[n] = wpv[n] = V3{0.0f, 0.0f, 0.0f};
        if (idx < WX * WY && gx >= 0 && gx < c.nx && gy >= 0 && gy < c.ny) {
            const int g = gy * c.nx + gx;
            wr[n] = ld3o(bf.r_in, N, g);
            ww[n] = ld3o(bf.w_in, N, g);
            if (k > 0) wsv[n] = ld3o(bf.s_in, N, g);
            if (jac) wpv[n] = ld3o(c.pinv, N, g);
        }
    }
    V3 pold = {0.0f, 0.0f, 0.0f}, x = pold, rk = pold, pv = pold;
    if (own) {
        if (k > 0) pold = ld3o(c.d1, N, i);
        x = ld3o(c.dv, N, i);
        rk = ld3o(bf.r_in, N, i);
        if (jac) pv = ld3o(c.pinv, N, i);
    }
    uint32_t mask = 0;
    if constexpr (STENCIL) mask = own ? ldo(c.pair_mask, (uint32_t)i) : 0u;
    const bool pinned = own ? ldo(c.pin, (uint32_t)i) != 0 : true;

    // ---- gamma_k, delta_k (the same lane tree as the other launches)
    if (threadIdx.x < 64) {
        float sg = 0.0f, sd = 0.0f;
#pragma unroll
        for (int j = 0; j < NP; j++) {
            sg += pg[j];
            sd += pd[j];
        }
        for (int t = threadIdx.x + 64 * NP; t < nt; t += 64) {
            sg += c.del_part[(size_t)k * nt + t];
            sd += c.sig_part[(size_t)k * nt + t];
        }
        sg = wave_sum(sg);
        sd = wave_sum(sd);
        if (threadIdx.x == 0) {
            sh.bc = sg;
            sh.bc2 = sd;
        }
    }
    __syncthreads();
    if (done) return;
    const float gamma = sh.bc, delta = sh.bc2;
    const float thresh = s.tol_mode == 1 ? s.tol2 * (k == 0 ? gamma : gamma0) : s.tol2;
    const bool stop = s.tol_mode != 2 && !(gamma > thresh);
    const float beta = (k > 0 && gamma_old != 0.0f) ? gamma / gamma_old : 0.0f;
    float den = delta;
    if (beta != 0.0f && alpha_old != 0.0f) {
        float t = beta * gamma;
        t = t / alpha_old;
        den = delta - t;
    }
    const bool brk = !stop && (den < 0.0f || !isfinite(den));
    const float alpha = den == 0.0f ? 0.0f : gamma / den;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c.scal[k] = gamma;
        c.scal[c.cg1_alpha + k] = alpha;
        if (stop || brk) {
            c.ctl[0] = 1;
            c.ctl[1] = k;
            if (brk) c.ctl[2] |= OC_SOLVE_BREAKDOWN;
        }
    }
    if (stop || brk) return;

    // ---- pair blocks of this vertex (the SpMV below)
    constexpr int NS = STENCIL ? kStencil : WP;
    uint16_t m[NS];
    float C[NS][6];
    if constexpr (STENCIL) {
#pragma unroll
        for (int q = 0; q < kStencil; q++) {
            const int di = stencil_di(q), dj = stencil_dj(q);
            const uint32_t blk = stencil_owner(q) ? (uint32_t)i : (uint32_t)(i + dj * c.nx + di);
            const uint32_t off = blk + (uint32_t)c.stencil_plane[q] * 6u * (uint32_t)N;
#pragma unroll
            for (int e = 0; e < 6; e++) C[q][e] = ((mask >> q) & 1u) ? ldo(c.blocks, off + (uint32_t)(e * N)) : 0.0f;
        }
    } else {
#pragma unroll
        for (int sl = 0; sl < WP; sl++) {
            m[sl] = (own && sl < c.wp) ? ldo(c.pair_m, (uint32_t)(sl * N + i)) : kEmptySlot;
            if (m[sl] != kEmptySlot) {
                const int j = i + slot_dj(m[sl]) * c.nx + slot_di(m[sl]);
                const int blk = ((m[sl] >> 12) & 1) ? i : j;
                const uint32_t b0 = (uint32_t)((m[sl] >> 8) & 15) * 6u * (uint32_t)N + (uint32_t)blk;
#pragma unroll
                for (int e = 0; e < 6; e++) C[sl][e] = ldo(c.blocks + (size_t)e * N, b0);
            } else {
#pragma unroll
                for (int e = 0; e < 6; e++) C[sl][e] = 0.0f;
            }
        }
    }

    // ---- s_k, r_{k+1}, u_{k+1} on the tile + halo; the tile's own values out
#pragma unroll
    for (int n = 0; n < NWIN; n++) {
        const int idx = threadIdx.x + n * NT;
        if (idx < WX * WY) {
            const int wx = idx % WX, wy = idx / WX;
            const V3 sk = k == 0 ? ww[n] : V3{ww[n].x + beta * wsv[n].x, ww[n].y + beta * wsv[n].y,
                                              ww[n].z + beta * wsv[n].z};
            const V3 rn = {wr[n].x - alpha * sk.x, wr[n].y - alpha * sk.y, wr[n].z - alpha * sk.z};
            const V3 un = jac ? V3{wpv[n].x * rn.x, wpv[n].y * rn.y, wpv[n].z * rn.z} : rn;
            const int gx = x0 + wx, gy = y0 + wy;
            if (wx >= H && wx < H + TX && wy >= H && wy < H + TY && gx < c.nx && gy < c.ny) {
                const int g = gy * c.nx + gx;
                st3o(bf.s_out, N, g, sk);
                st3o(bf.r_out, N, g, rn);
            }
            if (wx >= H && wx < H + TX && wy >= H && wy < H + TY) {
                sh.rt[0][wy - H][wx - H] = rn.x;
                sh.rt[1][wy - H][wx - H] = rn.y;
                sh.rt[2][wy - H][wx - H] = rn.z;
            }
            sh.wu[0][wy][wx] = un.x;
            sh.wu[1][wy][wx] = un.y;
            sh.wu[2][wy][wx] = un.z;
        }
    }
    // this vertex: p_k = u_k + beta p_{k-1}, dv += alpha p_k
    if (own) {
        const V3 uk = jac ? V3{pv.x * rk.x, pv.y * rk.y, pv.z * rk.z} : rk;
        const V3 pk = k == 0 ? uk : V3{uk.x + beta * pold.x, uk.y + beta * pold.y, uk.z + beta * pold.z};
        st3o(c.d1, N, i, pk);
        st3o(c.dv, N, i, V3{x.x + alpha * pk.x, x.y + alpha * pk.y, x.z + alpha * pk.z});
    }
    __syncthreads();

    // ---- w_{k+1} = S A u_{k+1}; partials of r.u and w.u
    float tg = 0.0f, td = 0.0f;
    if (own) {
        const V3 ui = {sh.wu[0][ly + H][lx + H], sh.wu[1][ly + H][lx + H], sh.wu[2][ly + H][lx + H]};
        V3 acc = {s.md * ui.x, s.md * ui.y, s.md * ui.z};
        if constexpr (STENCIL) {
#pragma unroll
            for (int q = 0; q < kStencil; q++) {
                if (!((mask >> q) & 1u)) continue;
                const int wy = ly + H + stencil_dj(q), wx = lx + H + stencil_di(q);
                V3 w = {sh.wu[0][wy][wx] - ui.x, sh.wu[1][wy][wx] - ui.y, sh.wu[2][wy][wx] - ui.z};
                V3 a = symmv(C[q], w);
                acc = {acc.x + a.x, acc.y + a.y, acc.z + a.z};
            }
        } else {
#pragma unroll
            for (int sl = 0; sl < WP; sl++) {
                if (m[sl] == kEmptySlot) break;
                const int wy = ly + H + slot_dj(m[sl]), wx = lx + H + slot_di(m[sl]);
                V3 w = {sh.wu[0][wy][wx] - ui.x, sh.wu[1][wy][wx] - ui.y, sh.wu[2][wy][wx] - ui.z};
                V3 a = symmv(C[sl], w);
                acc = {acc.x + a.x, acc.y + a.y, acc.z + a.z};
            }
        }
        const V3 wn = pinned ? V3{0.0f, 0.0f, 0.0f} : acc;
        st3o(bf.w_out, N, i, wn);
        const V3 rn = {sh.rt[0][ly][lx], sh.rt[1][ly][lx], sh.rt[2][ly][lx]};
        tg = dot3(rn, ui);
        td = dot3(wn, ui);
    }
    const float pgs = tile_sum<NT>(tg, sh.ws);
    const float pds = tile_sum<NT>(td, sh.ws2);
    if (threadIdx.x == 0) {
        c.del_part[(size_t)(k + 1) * nt + tile] = pgs;
        c.sig_part[(size_t)(k + 1) * nt + tile] = pds;
    }
}

// CG iteration k, part 2: dv += alpha d, r -= alpha q, partial r.r.  Returns
// true when the solve has stopped (breakdown or an earlier stop).
template <int TX, int TY>
__device__ inline bool axpy_phase(const DevCloth& c, const StepScalars& s, int k, bool read_done,
                                  float* ws, float& bc, int vb) {
    constexpr int NT = TX * TY;
    const int nt = c.nt, N = c.N;
    const int tile = tile_of_block(vb, nt);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    const bool own = gi < c.nx && gj < c.ny;
    const int i = gj * c.nx + gi;

    // ---- loads that do not depend on alpha
    const int done = read_done ? c.ctl[0] : 0;
    const float delta = c.scal[k];
    float pv[kPartialRegs];
    if (threadIdx.x < 64) partial_load(c.sig_part + (size_t)k * nt, nt, pv);
    const float* dcur = (k & 1) ? c.d1 : c.d0;
    const bool jac = (s.flags & OC_FLAG_JACOBI) != 0;
    V3 d = {0.0f, 0.0f, 0.0f}, q = d, x = d, r = d, jv = d;
    if (own) {
        d = ld3o(dcur, N, i);
        q = ld3o(c.q, N, i);
        x = ld3o(c.dv, N, i);
        r = ld3o(c.r, N, i);
        if (jac) jv = ld3o(c.pinv, N, i);
    }
    if (threadIdx.x < 64) {
        const float sum = partial_finish(c.sig_part + (size_t)k * nt, nt, pv);
        if (threadIdx.x == 0) bc = sum;
    }
    __syncthreads();
    if (done) return true;
    const float sigma = bc;
    if (sigma < 0.0f || !isfinite(sigma)) {
        if (vb == 0 && threadIdx.x == 0) {
            c.ctl[0] = 1;
            c.ctl[1] = k;
            c.ctl[2] |= OC_SOLVE_BREAKDOWN;
        }
        return true;
    }
    // sigma == 0 only after r (hence d) underflowed: no update, no 0/0
    const float alpha = sigma == 0.0f ? 0.0f : delta / sigma;
    float t = 0.0f;
    if (own) {
        x = {x.x + alpha * d.x, x.y + alpha * d.y, x.z + alpha * d.z};
        r = {r.x - alpha * q.x, r.y - alpha * q.y, r.z - alpha * q.z};
        st3o(c.dv, N, i, x);
        st3o(c.r, N, i, r);
        if (jac) {
            const V3 z = {jv.x * r.x, jv.y * r.y, jv.z * r.z};
            st3o(c.s, N, i, z);
            t = dot3(r, z);
        } else {
            t = dot3(r, r);
        }
    }
    float p = tile_sum<NT>(t, ws);
    if (threadIdx.x == 0) c.del_part[(size_t)(k + 1) * nt + tile] = p;
    return false;
}

template <int TX, int TY>
__global__ __launch_bounds__(TX* TY) void k_cg_axpy(DevCloth c, StepScalars s, int k) {
    __shared__ float ws[TX * TY / 64];
    __shared__ float bc;
    axpy_phase<TX, TY>(c, s, k, true, ws, bc, blockIdx.x);
}

// ---------------------------------------------------------------------------
// resident CG: a whole solve in one launch, the pair blocks in registers
// ---------------------------------------------------------------------------
// Every block keeps a region of TX x (TY VT) vertices for the whole solve:
// each thread holds VT vertices' pair blocks, r, q and solution in registers
// and the region's d with its halo sits in LDS, so an iteration reads no
// matrix and no vector from memory.  What blocks tell each other goes
// through memory as 8-byte words (value, tag) that are stored and polled with
// relaxed device-scope accesses: a word is its own flag, so no fence (which
// on MI355X writes back the XCD's L2) and no barrier counter is needed.
// Two exchanges per iteration, as the recurrence has two reductions:
//   alpha : the tiles' d.q partials
//   beta  : the tiles' r.z partials, and z of the region's outer two rows and
//           columns, from which the neighbours form their halo's d
// The tag of exchange n of a solve is the solve's epoch base + n + 1.  A block
// publishes exchange n + 1 only after it has read all of exchange n, and
// every exchange needs every block's partials; so when a block publishes
// n + 2 all have read n, and two sets of partials and one set of rims are
// enough.  Partials are stored once per XCD (8 copies, 8 lanes) in tile
// order, and a block polls its own XCD's copy.
// The partials are summed in tile order exactly as the per-iteration launches
// sum them.
//
// The blocks wait for each other, so they must run at the same time.  They
// are launched one per CU at most, but another stream's or process's work may
// hold some CUs: thread 0 of each block signs in, and the blocks take the
// resident path once all have.  If they have not within kRollCallTicks, the
// roll is closed, and every block, those that start later too, runs tiles of
// the per-iteration phases below, by tickets, until the solve is done.  So the
// launch needs no cooperative launch (20 us each, measured) and cannot wait
// for a block that never starts.
//
// Measured per iteration (30 to 40 iterations, two launches per iteration
// before): 512x512 16.3 -> 7.7 us, 256x256 about 9 -> 4.4, 128x128 9.7 -> 3.9,
// 21x21 7.1 -> 3.4.  An exchange takes 1.0 us between a few blocks and 1.7 to
// 2.4 us among 256 (store to the coherence point, then polled loads of 512
// words); the rest at 512x512, about 3 us, is the arithmetic: 16 waves per CU
// issue about 340 vector instructions each per iteration, 29% of the issue
// slots of the whole solve.
constexpr int kPollLimit = 1 << 21;              // polls of one exchange (seconds)

// Grid barrier of the persistent solve's blocks: every block adds 1 to *bar and waits until it reaches target.  The add is a
// release (the block's writes reach the device-coherent level first); the
// wait polls with relaxed agent-scope loads, which read the coherent value
// without invalidating caches, and a single acquire fence follows.  The wait
// is bounded; on time-out the block sets ctl[4] and the caller ends the
// kernel, so every wave exits.
__device__ inline bool grid_barrier(unsigned* bar, unsigned target, int* err) {
    __syncthreads();
    __shared__ int ok;
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(bar, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        int good = 1;
        unsigned spins = 0;
        while (__hip_atomic_load(bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            __builtin_amdgcn_s_sleep(1);
            if (++spins > (1u << 24)) {
                good = 0;
                __hip_atomic_fetch_or(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        ok = good;
    }
    __syncthreads();
    return ok != 0;
}

// All CG iterations in one cooperative launch, for any topology: the spmv and
// axpy phases of the multi-kernel form, separated by grid barriers instead of
// kernel boundaries.  Each resident block serves tiles blockIdx.x,
// + gridDim.x, ... with the same per-tile code.  Every block owns at least one
// tile and so takes the same stop decisions as the others: all blocks pass the
// same barriers.
template <int TX, int TY, int WP>
__global__ __launch_bounds__(TX* TY) void k_cg_persistent(DevCloth c, StepScalars s, unsigned* bar) {
    __shared__ SpmvShared<TX, TY> sh;
    __shared__ float ws[TX * TY / 64];
    __shared__ float bc;
    const unsigned nb = gridDim.x;
    unsigned target = 0;
    for (int k = 0; k < s.max_it; k++) {
        bool stop = false;
        for (int vb = blockIdx.x; vb < c.nt && !stop; vb += gridDim.x)
            stop = spmv_phase<TX, TY, WP>(c, s, k, false, sh, vb);
        if (stop) break;
        target += nb;
        if (!grid_barrier(bar, target, c.ctl + 4)) break;
        for (int vb = blockIdx.x; vb < c.nt && !stop; vb += gridDim.x)
            stop = axpy_phase<TX, TY>(c, s, k, false, ws, bc, vb);
        if (stop) break;
        target += nb;
        if (!grid_barrier(bar, target, c.ctl + 4)) break;
    }
}

// The same phases of a cloth in the stencil form, G tiles per ticket (what a
// block of a complete team would have, for as few tickets as serve it), by
// however many blocks there are (of at least TX * TY threads each, the first
// of which work).  A phase that stops does so in every tile, and the block
// that has its tile 0 writes the control words and, with finish, the status.
template <int TX, int TY, int G>
__device__ inline void cg_tickets(const DevCloth& c, const StepScalars& s, bool finish, SpmvShared<TX, TY>& sh, float* ws,
                                  float& bc, Ticket& t) {
    unsigned* const q = c.sync + kSyncTickets;
    const unsigned pieces = (unsigned)(c.nt + G - 1) / G;  // at most 256, of 2 * 100000 phases
    const unsigned total = 2u * (unsigned)s.max_it * pieces;
    for (;;) {
        const int what = ticket_take(q, pieces, total, c.ctl, c.ctl + 4, t);
        if (what == kTicketOver) return;
        if (what == kTicketLast) break;
        const int phase = (int)(t.n / pieces), v0 = (int)(t.n % pieces) * G;
        bool stop = false;
#pragma unroll 1
        for (int vb = v0; vb < min(v0 + G, c.nt) && !stop; vb++) {
            if (vb > v0) __syncthreads();  // (the shared memory of the tile before)
            stop = (phase & 1) ? axpy_phase<TX, TY>(c, s, phase >> 1, false, ws, bc, vb)
                               : spmv_phase<TX, TY, kStencil, true, true>(c, s, phase >> 1, false, sh, vb);
        }
        ticket_done(q);
        if (!stop) continue;
        if (v0 != 0) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // (thread 0 has written what all read now)
        break;
    }
    __syncthreads();
    if (finish) cg_finish_block(c, s, &bc);
}

// Region r of block b: blocks go to XCDs round-robin and each XCD takes a
// contiguous run of regions.
__device__ inline int region_of_block(int b, int nb) {
    const int x = b & 7, q = nb >> 3, r = nb & 7;
    return x * q + min(x, r) + (b >> 3);
}

// HY rows per region, one thread per vertex.  An iteration evaluates every
// pair once: a vertex computes a = C (d_j - d_i) of the six pairs it owns
// (those owned outside the region whose partner is inside, the strips, are
// computed by the last threads) and leaves them in LDS, where the partner
// takes them negated; swapping a pair's ends negates w and a exactly, and
// both ends add in stencil order, so the sums are the SpMV's bits (as in
// the spring-once assembly).  That halves the arithmetic and the registers
// for blocks (36 floats) against every vertex computing its 12 pairs.
// Component planes in LDS are whole multiples of 64 words apart, so that two
// components move in one LDS instruction without bank conflicts.
template <int TX, int HY>
struct ResidentShared {
    static constexpr int WX = TX + 2 * H, WY = HY + 2 * H, NT = TX * HY;
    static constexpr int NS = (strip_total<TX, HY>() + 63) / 64 * 64;  // strip pairs, padded
    static constexpr int WP = (WX * WY + 63) / 64 * 64;
    float wd[3][WP];                // d on the region and its halo (z between two iterations)
    float res[3][kOwned * NT + NS];  // a of the owned pairs, direction by direction, then the strips'
    float sc[6][NS];                // the strip pairs' blocks
    float x[3][NT];                 // the solution
    float ws[NT / 64];
    float bc;       // alpha or beta of the exchange just read
    int go;         // kGo, kStop, kBreakdown or kTimeout, after the same exchange
    int late;       // a halo vertex's z did not come
    int team;
};
constexpr int kTeamAll = 0, kTeamOpen = 1, kTeamOver = 2;
constexpr int kGo = 0, kStop = 1, kBreakdown = 2, kTimeout = 4;

// Up to here two assembly blocks per tile have a CU each.
constexpr int kRowTiles = 128;
static_assert(kRowTiles <= 64 * kPartialRegs, "the rows are combined into a solve's first loads");
// A tile's partial of r.z from its rows' sums, as tile_sum adds them, and
// partial_load of them (nt <= kRowTiles).
__device__ inline float row_partial(const DevCloth& c, int tile) {
    const float* q = c.row_part + tile * kTileY;
    float w[kTileY];
#pragma unroll
    for (int k = 0; k < kTileY; k++) w[k] = q[k];
    float p = w[0];
#pragma unroll
    for (int k = 1; k < kTileY; k++) p = p + w[k];
    return p;
}
__device__ inline void row_partial_load(const DevCloth& c, float* v) {
#pragma unroll
    for (int j = 0; j < kPartialRegs; j++) {
        const int k = threadIdx.x + 64 * j;
        v[j] = 64 * j < kRowTiles && k < c.nt ? row_partial(c, k) : 0.0f;
    }
}

template <int TX, int HY>
__global__ __launch_bounds__(TX* HY) void k_cg_resident(DevCloth c, StepScalars s, int nb, int finish) {
    constexpr int TY = kTileY, VT = HY / TY;            // tiles per region
    constexpr int NT = TX * HY, NWT = TX * TY / 64;     // threads; waves per tile
    using SH = ResidentShared<TX, HY>;
    constexpr int WX = SH::WX;
    constexpr int E = resident_rim(TX, HY);             // rim entries of a region
    constexpr int NH = 2 * H * TX + 2 * H * HY + 4;     // halo vertices read by the stencil
    constexpr int NJ = kResidentTiles / 64;             // partials per lane of wave 0
    constexpr int S0 = NT - SH::NS;                     // first strip thread
    static_assert(TX == 64 && HY % TY == 0, "one row per wave, whole tiles");
    static_assert(E <= NH && NH <= NT - 64 && S0 >= 0, "rims and halo by waves 1.., strips by the last waves");
    union Shared {
        SH r;
        struct {
            SpmvShared<TX, TY> sp;
            float ws[NWT];
            float bc;
            Ticket ticket;
        } t;
    };
    __shared__ Shared lds;
    SH& sh = lds.r;
    const int tid = threadIdx.x, lx = tid % TX, ly = tid / TX;
    // sign in, unless the solve is already done (a second solve of one
    // assembly, or a block that starts after the others have finished it)
    int done = 0;
    if (tid == 0 && !(done = c.ctl[0])) roll_call_sign(c.sync + 1);

    const int N = c.N, nx = c.nx, ny = c.ny, ntx = c.ntx;
    const int reg = region_of_block(blockIdx.x, nb);
    const int rx = reg % ntx, ry = reg / ntx;
    const int x0 = rx * TX, y0 = ry * HY;
    const int gi = x0 + lx, gj = y0 + ly, i = gj * nx + gi;
    const bool own = gi < nx && gj < ny;
    const bool jac = (s.flags & OC_FLAG_JACOBI) != 0;
    const unsigned base = c.sync[0];

    // ---- this thread's vertex: mask, vectors, owned blocks
    const uint32_t mask = own ? ldo(c.pair_mask, (uint32_t)i) : 0u;
    float pv[kPartialRegs];
    if (tid < 64) {
        if (VT == 1 && c.asm_rows)
            row_partial_load(c, pv);
        else
            partial_load(c.del_part, c.nt, pv);
    }
    V3 r = {0.0f, 0.0f, 0.0f}, pn = r, d = r;
    bool pinned = true;
    if (own) {
        r = ld3o(c.r, N, i);
        const V3 x = ld3o(c.dv, N, i);
        sh.x[0][tid] = x.x;
        sh.x[1][tid] = x.y;
        sh.x[2][tid] = x.z;
        d = ld3o(c.d0, N, i);
        if (jac) pn = ld3o(c.pinv, N, i);
        pinned = ldo(c.pin, (uint32_t)i) != 0;
    }
    auto block_of = [&](float (&C)[6], int plane, int g, bool have) {
        const uint32_t off = (uint32_t)g + (uint32_t)plane * 6u * (uint32_t)N;
#pragma unroll
        for (int q = 0; q < 6; q++) C[q] = have ? ldo(c.blocks, off + (uint32_t)(q * N)) : 0.0f;
    };
    float C[kOwned][6];
#pragma unroll
    for (int o = 0; o < kOwned; o++) block_of(C[o], c.stencil_plane[owned_k(o)], i, (mask >> owned_k(o)) & 1u);
    // where the partner of this vertex's pairs finds the owner's a (two
    // 16-bit places per register)
    unsigned place[kOwned / 2] = {};
#pragma unroll
    for (int o = 0; o < kOwned; o++) {
        const int wx = lx - own_dx(o), wy = ly - own_dy(o);
        const int w = (wx >= 0 && wx < TX && wy >= 0)
                          ? o * NT + wy * TX + wx
                          : kOwned * NT + strip_base<TX, HY>(o) + strip_index<TX, HY>(o, wx, wy);
        place[o / 2] |= (unsigned)w << (16 * (o & 1));
    }
    // this thread's strip pair: the owner's window entry and its partner's
    int sown = 0, spar = 0;
    bool strip = false;
    if (tid >= S0 && tid - S0 < strip_total<TX, HY>()) {
        int o, q, wx, wy;
        strip_of_column<TX, HY>(tid - S0, o, q);
        strip_owner<TX, HY>(o, q, wx, wy);
        const int gx = x0 + wx, gy = y0 + wy, g = gy * nx + gx;
        strip = gx >= 0 && gx < nx && gy >= 0 && gy < ny && ((ldo(c.pair_mask, (uint32_t)g) >> owned_k(o)) & 1u);
        sown = (wy + H) * WX + wx + H;
        spar = sown + own_dy(o) * WX + own_dx(o);
        float SC[6];
        block_of(SC, c.stencil_plane[owned_k(o)], g, strip);
#pragma unroll
        for (int e = 0; e < 6; e++) sh.sc[e][tid - S0] = SC[e];
    }
    // this thread's halo vertex: where its d lives in the window, and the rim
    // entry its owner publishes z in
    int hx = 0, hy = 0, hreg = 0, hent = 0;
    bool halo = false;
    if (const int e = tid - 64; e >= 0 && e < NH) {
        if (e < 2 * TX) {  // two rows above
            hx = e % TX, hy = e / TX - 2;
            hreg = reg - ntx, hent = 2 * TX + e;
        } else if (e < 4 * TX) {  // two rows below
            hx = e % TX, hy = HY + e / TX - 2;
            hreg = reg + ntx, hent = e - 2 * TX;
        } else if (e < 4 * TX + 2 * HY) {  // two columns left
            const int q = e - 4 * TX;
            hx = q / HY - 2, hy = q % HY;
            hreg = reg - 1, hent = 4 * TX + 2 * HY + q;
        } else if (e < 4 * TX + 4 * HY) {  // two columns right
            const int q = e - 4 * TX - 2 * HY;
            hx = TX + q / HY, hy = q % HY;
            hreg = reg + 1, hent = 4 * TX + q;
        } else {  // the four corners next to the region
            const int q = e - 4 * TX - 4 * HY;
            hx = (q & 1) ? TX : -1, hy = (q & 2) ? HY : -1;
            hreg = reg + ((q & 1) ? 1 : -1) + ((q & 2) ? ntx : -ntx);
            hent = ((q & 2) ? 0 : 3 * TX) + ((q & 1) ? 0 : TX - 1);
        }
        const int gx = x0 + hx, gy = y0 + hy;
        halo = gx >= 0 && gx < nx && gy >= 0 && gy < ny;
    }
    const int hw = (hy + H) * WX + hx + H;
    V3 hd = {0.0f, 0.0f, 0.0f}, hz = hd;
    if (halo) hd = ld3o(c.d0, N, (y0 + hy) * nx + x0 + hx);
    // this thread's rim entry: the window cell whose z it publishes
    int rw = 0;
    if (const int e = tid - 64; e >= 0 && e < E) {
        const int q = e - 4 * TX, qx = q / HY;
        rw = e < 4 * TX ? ((e < 2 * TX ? e / TX : HY - 4 + e / TX) + H) * WX + e % TX + H
                        : (q % HY + H) * WX + (qx < H ? qx : TX - 2 * H + qx) + H;
    }
    uint64_t* const rim = c.xch + resident_part_words(c.xstride);
    const unsigned hsrc = (unsigned)(hreg * 3 * E + hent), rout = (unsigned)(reg * 3 * E);
    // this XCD's copy of the tiles' partials
    unsigned xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    const uint64_t* const near = c.xch + (size_t)(xcc & 7u) * c.xstride;

    // Sum of the tiles' partials of exchange n (wave 0): polled until every
    // tag is the exchange's, then added as partial_finish does.
    auto poll_sum = [&](unsigned n, float& sum) -> bool {
        const uint64_t* p = near + (n & 1u) * c.xslots;
        const unsigned tag = base + n + 1u;
        uint64_t w[NJ];
        for (int spin = 0;; spin++) {
            bool ok = true;
#pragma unroll
            for (int j = 0; j < NJ; j++)
                w[j] = tid + 64 * j < c.nt ? xch_load(p, (unsigned)(tid + 64 * j)) : (uint64_t)tag << 32;
#pragma unroll
            for (int j = 0; j < NJ; j++) ok = ok && (unsigned)(w[j] >> 32) == tag;
            if (__all(ok)) break;
            if (spin > kPollLimit) return false;
        }
        float t = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; j++) t += __uint_as_float((unsigned)w[j]);
        sum = wave_sum(t);
        return true;
    };
    // The tiles' sums of t (tile_sum's order), published as exchange n.
    auto publish = [&](unsigned n, float t) {
        const float w = wave_sum(t);
        if ((tid & 63) == 0) sh.ws[tid >> 6] = w;
        __syncthreads();
        if (tid < 8 * VT && ry * VT + (tid >> 3) < c.nty) {  // 8 copies of each tile's partial
            const float* const q = sh.ws + (tid >> 3) * NWT;
            float p = q[0];
#pragma unroll
            for (int k = 1; k < NWT; k++) p = p + q[k];
            xch_store(c.xch, (tid & 7) * c.xstride + (n & 1u) * c.xslots + (ry * VT + (tid >> 3)) * ntx + rx, base + n + 1u,
                      p);
        }
    };
    // ---- d0 on the region and its halo; r.z of the start
    const int cw = (ly + H) * WX + lx + H;
    auto put = [&](int w, V3 v) {
        sh.wd[0][w] = v.x;
        sh.wd[1][w] = v.y;
        sh.wd[2][w] = v.z;
    };
    auto get = [&](int w) { return V3{sh.wd[0][w], sh.wd[1][w], sh.wd[2][w]}; };
    put(cw, d);
    if (halo) put(hw, hd);
    // r.z of the iteration at hand and of the one before, the stopping test's
    // threshold: kept by thread 0, which decides for the block (every block's
    // thread 0 decides alike) and hands on alpha and beta
    float delta = 0.0f, delta_old = 0.0f, delta0 = 0.0f, thresh = 0.0f;
    auto stopped = [&]() { return s.tol_mode != 2 && !(delta > thresh); };
    if (tid < 64) {
        delta = delta0 = partial_finish(c.del_part, c.nt, pv);
        thresh = s.tol_mode == 1 ? s.tol2 * delta0 : s.tol2;
    }
    if (tid == 0) {
        sh.go = stopped() ? kStop : kGo;
        sh.late = 0;
        sh.team = done ? kTeamOver : roll_call_wait(c.sync + 1, nb) ? kTeamAll : kTeamOpen;
    }
    __syncthreads();
    const int team = sh.team;
    if (team == kTeamOver) return;
    if (team == kTeamOpen) {
        __syncthreads();  // (the shared words above have been read)
        if (VT == 1 && c.asm_rows) {  // every block for itself, all the same
            for (int k = tid; k < c.nt; k += NT) c.del_part[k] = row_partial(c, k);
            __syncthreads();
        }
        if (tid < TX * TY) cg_tickets<TX, TY, VT>(c, s, finish != 0, lds.t.sp, lds.t.ws, lds.t.bc, lds.t.ticket);
        return;
    }

    // ---- iterations
    const bool full = __all(mask == 0xFFFu);  // every lane of the wave has all 12 neighbours
    int it = s.max_it, go = sh.go;
    float beta = 0.0f;
    for (int k = 0; k < s.max_it; k++) {
        if (go != kGo) {
            it = k;
            break;
        }
        if (k > 0) {  // d = z + beta d
            const V3 z = jac ? V3{pn.x * r.x, pn.y * r.y, pn.z * r.z} : r;
            d = {z.x + beta * d.x, z.y + beta * d.y, z.z + beta * d.z};
            put(cw, d);
            if (halo) {
                hd = {hz.x + beta * hd.x, hz.y + beta * hd.y, hz.z + beta * hd.z};
                put(hw, hd);
            }
            __syncthreads();
        }
        // q = S A d: the owned pairs, then every vertex's sum.  Pairs that do
        // not exist have a zero block; what they give is not added.
        V3 a[kOwned];
#pragma unroll
        for (int o = 0; o < kOwned; o++) a[o] = get(cw + own_dy(o) * WX + own_dx(o));
#pragma unroll
        for (int o = 0; o < kOwned; o++) {
            a[o] = symmv(C[o], V3{a[o].x - d.x, a[o].y - d.y, a[o].z - d.z});
            sh.res[0][o * NT + tid] = a[o].x;
            sh.res[1][o * NT + tid] = a[o].y;
            sh.res[2][o * NT + tid] = a[o].z;
        }
        if (strip) {
            const int t = tid - S0;
            const V3 e = get(sown), f = get(spar);
            float SC[6];
#pragma unroll
            for (int q = 0; q < 6; q++) SC[q] = sh.sc[q][t];
            const V3 b = symmv(SC, V3{f.x - e.x, f.y - e.y, f.z - e.z});
            sh.res[0][kOwned * NT + t] = b.x;
            sh.res[1][kOwned * NT + t] = b.y;
            sh.res[2][kOwned * NT + t] = b.z;
        }
        __syncthreads();
        V3 acc = {s.md * d.x, s.md * d.y, s.md * d.z};
        V3 p[kOwned];
#pragma unroll
        for (int o = 0; o < kOwned; o++) {
            const unsigned w = (here(place[o / 2]) >> (16 * (o & 1))) & 0xFFFFu;
            p[o] = {sh.res[0][w], sh.res[1][w], sh.res[2][w]};
        }
        auto add = [&](int kk) {
            const int o = owned_index(kk);
            return stencil_owner(kk) ? V3{acc.x + a[o].x, acc.y + a[o].y, acc.z + a[o].z}
                                     : V3{acc.x - p[o].x, acc.y - p[o].y, acc.z - p[o].z};
        };
        if (full) {
#pragma unroll
            for (int kk = 0; kk < kStencil; kk++) acc = add(kk);
        } else {
#pragma unroll
            for (int kk = 0; kk < kStencil; kk++) {
                const V3 n = add(kk);
                const bool have = (mask >> kk) & 1u;
                acc = {have ? n.x : acc.x, have ? n.y : acc.y, have ? n.z : acc.z};
            }
        }
        const V3 q = pinned ? V3{0.0f, 0.0f, 0.0f} : acc;
        publish(2u * k, own ? dot3(d, q) : 0.0f);
        if (tid < 64) {
            float sigma = 0.0f;
            const bool got = poll_sum(2u * k, sigma);
            // sigma == 0 only after r (hence d) underflowed: no update, no 0/0
            const float alpha = sigma == 0.0f ? 0.0f : delta / sigma;
            if (tid == 0) {
                sh.bc = alpha;
                sh.go = !got ? kTimeout : sigma < 0.0f || !isfinite(sigma) ? kBreakdown : kGo;
            }
        }
        __syncthreads();
        const float alpha = sh.bc;
        go = sh.go;
        if (go != kGo) {
            it = k;
            break;
        }
        const bool last = k + 1 == s.max_it;
        r = {r.x - alpha * q.x, r.y - alpha * q.y, r.z - alpha * q.z};
        const V3 z = jac ? V3{pn.x * r.x, pn.y * r.y, pn.z * r.z} : r;
        put(cw, z);
        publish(2u * k + 1u, own ? dot3(r, z) : 0.0f);
        const unsigned tag = base + 2u * k + 2u;
        if (!last && tid >= 64 && tid < 64 + E) {
            const V3 v = get(rw);
            const unsigned e = rout + tid - 64;
            xch_store(rim, e, tag, v.x);
            xch_store(rim, e + E, tag, v.y);
            xch_store(rim, e + 2 * E, tag, v.z);
        }
        sh.x[0][tid] = sh.x[0][tid] + alpha * d.x;
        sh.x[1][tid] = sh.x[1][tid] + alpha * d.y;
        sh.x[2][tid] = sh.x[2][tid] + alpha * d.z;
        if (last && blockIdx.x != 0) break;  // nothing more is read: block 0 records the status
        if (tid < 64) {
            float sum = 0.0f;
            const bool got = poll_sum(2u * k + 1u, sum);
            delta_old = delta;
            delta = sum;
            // beta = 0 once r.r has underflowed to 0 (fixed iteration counts)
            const float b = delta_old != 0.0f ? delta / delta_old : 0.0f;
            if (tid == 0) {
                sh.bc = b;
                sh.go = !got ? kTimeout : stopped() ? kStop : kGo;
            }
        } else if (halo && !last) {
            uint64_t w[3];
            for (int spin = 0;; spin++) {
#pragma unroll
                for (int e = 0; e < 3; e++) w[e] = xch_load(rim, hsrc + e * E);
                if ((unsigned)(w[0] >> 32) == tag && (unsigned)(w[1] >> 32) == tag && (unsigned)(w[2] >> 32) == tag)
                    break;
                if (spin > kPollLimit) {
                    sh.late = 1;
                    break;
                }
            }
            hz = {__uint_as_float((unsigned)w[0]), __uint_as_float((unsigned)w[1]), __uint_as_float((unsigned)w[2])};
        }
        // (a stop after the last iteration leaves it = max_it)
        __syncthreads();
        beta = sh.bc;
        go = sh.late ? kTimeout : last ? sh.go & kTimeout : sh.go;
    }

    // The next solve's tags start past those that were used, which every block
    // has written over the older ones in the words (a solve that stops at once
    // uses none; were the start to move on all the same, it could come round to
    // tags that the words still hold).
    if (go == kTimeout) {  // an exchange timed out: report it, leave dv as it was
        if (tid == 0) {
            __hip_atomic_fetch_or(c.ctl + 4, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (blockIdx.x == 0) {
                c.ctl[0] = 1;
                c.sync[3] = base + 2u * (unsigned)it + 2u;
            }
        }
        return;
    }
    if (own) st3o(c.dv, N, i, V3{sh.x[0][tid], sh.x[1][tid], sh.x[2][tid]});
    if (blockIdx.x == 0 && tid == 0) {
        // as a stopped solve of the per-iteration launches leaves them; the
        // status bits follow as cg_finish_block derives them
        c.scal[0] = delta0;
        c.scal[it] = delta;
        c.sync[3] = base + 2u * (unsigned)(go == kBreakdown ? it + 1 : it);
        c.ctl[0] = 1;
        c.ctl[1] = it;
        int st = c.ctl[2] | (go == kBreakdown ? OC_SOLVE_BREAKDOWN : 0);
        if (finish) {
            if (s.tol_mode != 2 && delta > thresh && !(st & OC_SOLVE_BREAKDOWN)) st |= OC_SOLVE_NOT_CONVERGED;
            if (!isfinite(delta)) st |= OC_SOLVE_NONFINITE;
            atomicOr(c.ctl + 3, st);
        }
        c.ctl[2] = st;
    }
}

__global__ void k_reset_barrier(unsigned* bar) {
    if (threadIdx.x == 0) *bar = 0u;
}

// Iteration count and status of the solve (one 64-thread block).
__global__ void k_cg_finish(DevCloth c, StepScalars s) {
    __shared__ float bc;
    cg_finish_block(c, s, &bc);
}

// v += dv, x += h v, optional ground clamp (IE:693-699).  FIN: block 0 also
// records the solve's iteration count and status (the step's last launch).
// BALL: then the collider, which puts a vertex on its surface and stops it
// (k_ellipsoid's work without a launch of its own).
template <bool FIN, bool BALL>
__global__ __launch_bounds__(256) void k_update(DevCloth c, StepScalars s, oc_ellipsoid e) {
    if (FIN && blockIdx.x == 0) {
        __shared__ float bc;
        cg_finish_block(c, s, &bc);
    }
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= c.N) return;
    const int N = c.N;
    V3 v = ld3o(c.v, N, i), dv = ld3o(c.dv, N, i), x = ld3o(c.x, N, i);
    v = {v.x + dv.x, v.y + dv.y, v.z + dv.z};
    x = {x.x + s.h * v.x, x.y + s.h * v.y, x.z + s.h * v.z};
    if ((s.flags & OC_FLAG_GROUND_CLAMP) && x.y < 0.0f) x.y = 0.0f;
    bool inside = false;
    V3 p = x;
    if constexpr (BALL) p = ellipsoid_push(e, x, inside);
    st3o(c.v, N, i, inside ? V3{0.0f, 0.0f, 0.0f} : v);
    st3o(c.x, N, i, p);
    if (!(isfinite(x.x) && isfinite(x.y) && isfinite(x.z) && isfinite(v.x) && isfinite(v.y) &&
          isfinite(v.z))) {
        atomicOr(c.ctl + 2, OC_SOLVE_NONFINITE);
        atomicOr(c.ctl + 3, OC_SOLVE_NONFINITE);
    }
}

// ---------------------------------------------------------------------------
// adjoint of one step
// ---------------------------------------------------------------------------
// Adjoint solve start: gvt = gv' + h gx', r = d = S gvt, mu = 0, partial r.r
template <int TX, int TY>
__global__ __launch_bounds__(TX* TY) void k_adj_init(DevCloth c, StepScalars s, AdjointBufs a) {
    constexpr int NT = TX * TY;
    __shared__ float ws[NT / 64];
    const int lx = threadIdx.x % TX, ly = threadIdx.x / TX;
    const int tile = tile_of_block(blockIdx.x, c.nt);
    const int bx = tile % c.ntx, by = tile / c.ntx;
    const int gi = bx * TX + lx, gj = by * TY + ly;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c.ctl[0] = 0;
        c.ctl[1] = 0;
        c.ctl[2] = 0;
    }
    float t = 0.0f;
    if (gi < c.nx && gj < c.ny) {
        const int N = c.N, i = gj * c.nx + gi;
        V3 gx = ld3(a.gx_out, N, i), gv = ld3(a.gv_out, N, i);
        V3 g = {gv.x + s.h * gx.x, gv.y + s.h * gx.y, gv.z + s.h * gx.z};
        st3(a.gvt, N, i, g);
        V3 r = c.pin[i] ? V3{0.0f, 0.0f, 0.0f} : g;
        st3(c.r, N, i, r);
        st3(c.dv, N, i, V3{0.0f, 0.0f, 0.0f});
        if (s.flags & OC_FLAG_JACOBI) {  // pinv from the re-assembly
            const V3 pv = ld3(c.pinv, N, i);
            const V3 z = {pv.x * r.x, pv.y * r.y, pv.z * r.z};
            st3(c.s, N, i, z);
            st3(c.d0, N, i, z);
            t = dot3(r, z);
        } else {
            st3(c.d0, N, i, r);
            t = dot3(r, r);
        }
    }
    float p = tile_sum<NT>(t, ws);
    if (threadIdx.x == 0) c.del_part[tile] = p;
}

// gx_in = gx' + dJ/dx, gv_in = gvt + dJ/dv, gks += dJ/dks (added by each
// spring's p1).  c.x, c.v: pre-step state; c.dv: the step's solution.  One
// wave per block, so that a cloth of 128x128 already has a wave on every CU:
// 15 us there, 43 when the slots, neighbours and constants of a spring were
// loaded one after the other by 512-thread blocks.  Bound by the issue of a
// wave's twelve springs, about 400 instructions each.
constexpr int kGatherThreads = 64;
__global__ __launch_bounds__(kGatherThreads) void k_adj_gather(DevCloth c, StepScalars s, AdjointBufs a) {
    const int N = c.N, i = blockIdx.x * kGatherThreads + threadIdx.x;
    if (i >= N) return;
    V3 gx = ld3(a.gx_out, N, i), gv = ld3(a.gvt, N, i);
    const V3 mi = ld3(a.mu, N, i);
    if (s.damp != 0.0f && !c.pin[i])  // the damping force c v_i: dJ/dv_i += h c mu_i
        gv = {gv.x + s.h * (s.damp * mi.x), gv.y + s.h * (s.damp * mi.y), gv.z + s.h * (s.damp * mi.z)};
    const AdjGatherIn in = {c.x, c.v, a.mu, c.dv, c.ainc_s, c.ainc_m, N, c.wa};
    adj_gather_springs(in, i, c.nx, s.h, s.hh,
                       [&](int, int sp, float& L0, float& ks, float& kd) {
                           L0 = c.L0[sp];
                           ks = c.ks[sp];
                           kd = c.kd[sp];
                       },
                       a.gks, gx, gv);
    st3(a.gx_in, N, i, gx);
    st3(a.gv_in, N, i, gv);
}

// Three vectors of n quads of floats into dst, one after the other.
__global__ __launch_bounds__(256) void k_keep_state(const float4* x, const float4* v, const float4* dv, float4* dst,
                                                    unsigned n) {
    const unsigned t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const float4 a = x[t], b = v[t], c = dv[t];
    dst[t] = a;
    dst[n + t] = b;
    dst[2 * (size_t)n + t] = c;
}

thread_local LaunchProfile* t_prof = nullptr;

// Launch with the installed profile's next event pair, if any (see
// LaunchProfile).
template <typename F, typename... Args>
hipError_t launch_k(int kind, F kernel, dim3 grid, dim3 block, hipStream_t st, Args... args) {
    LaunchProfile* p = t_prof;
    if (p && p->n < p->cap) {
        const int k = p->n++;
        p->kind[k] = kind;
        hipExtLaunchKernelGGL(kernel, grid, block, 0, st, p->start[k], p->stop[k], 0, args...);
    } else {
        hipLaunchKernelGGL(kernel, grid, block, 0, st, args...);
    }
    return hipGetLastError();
}

}  // namespace

void set_launch_profile(LaunchProfile* p) { t_prof = p; }

hipError_t launch_adj_init(const DevCloth& c, const StepScalars& s, const AdjointBufs& a,
                           hipStream_t st) {
    hipLaunchKernelGGL((k_adj_init<kTileX, kTileY>), dim3(c.nt), dim3(kTileX * kTileY), 0, st, c, s,
                       a);
    return hipGetLastError();
}

hipError_t launch_adj_gather(const DevCloth& c, const StepScalars& s, const AdjointBufs& a,
                             hipStream_t st) {
    hipLaunchKernelGGL(k_adj_gather, dim3((c.N + kGatherThreads - 1) / kGatherThreads), dim3(kGatherThreads), 0, st, c,
                       s, a);
    return hipGetLastError();
}

hipError_t launch_keep_state(const float* x, const float* v, const float* dv, float* dst, size_t floats,
                             hipStream_t st) {
    if (floats % 4 != 0 || floats > (size_t)UINT32_MAX) return hipErrorInvalidValue;
    const unsigned n = (unsigned)(floats / 4);
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_keep_state, dim3((n + 255) / 256), dim3(256), 0, st, (const float4*)x, (const float4*)v,
                       (const float4*)dv, (float4*)dst, n);
    return hipGetLastError();
}

hipError_t launch_forces(const DevCloth& c, const StepScalars& s, hipStream_t st) {
    hipLaunchKernelGGL((k_forces<kTileX, kTileY>), dim3(c.nt), dim3(kTileX * kTileY), 0, st, c, s);
    return hipGetLastError();
}

hipError_t launch_assemble(const DevCloth& c, const StepScalars& s, hipStream_t st, bool fused_update) {
    // A fused update needs a warm start (a cold assembly zeroes dv, which
    // neighbouring blocks still read for the update) and at least one CG
    // iteration (the previous solve's status is taken from partials that a
    // solve without iterations leaves where this assembly writes its own).
    if (fused_update && (!s.warm || s.max_it < 1)) return hipErrorInvalidValue;
    const dim3 grid(c.nt), block(kTileX * kTileY);
    if (c.asm_rows) {
        const dim3 half(c.ntx * ((c.ny + kTileY / 2 - 1) / (kTileY / 2))), hb(kTileX * kTileY / 2);
        return fused_update ? launch_k(0, k_assemble_pairs<kTileX, kTileY / 2, true>, half, hb, st, c, s)
                            : launch_k(0, k_assemble_pairs<kTileX, kTileY / 2, false>, half, hb, st, c, s);
    }
    if (c.stencil_asm)
        return fused_update ? launch_k(0, k_assemble_st<kTileX, kTileY, true>, grid, block, st, c, s)
                            : launch_k(0, k_assemble_st<kTileX, kTileY, false>, grid, block, st, c, s);
    if (c.wa <= 16)
        return fused_update ? launch_k(0, k_assemble<kTileX, kTileY, 16, true>, grid, block, st, c, s)
                            : launch_k(0, k_assemble<kTileX, kTileY, 16, false>, grid, block, st, c, s);
    return fused_update
               ? launch_k(0, k_assemble<kTileX, kTileY, kMaxAssemblyWidth, true>, grid, block, st, c, s)
               : launch_k(0, k_assemble<kTileX, kTileY, kMaxAssemblyWidth, false>, grid, block, st, c, s);
}

// cst[spring_cst[sp] + q*N] = (L0, ks, kd)[q][sp] for q in [q0, q0 + nq).
__global__ __launch_bounds__(256) void k_scatter_cst(DevCloth c, const int32_t* spring_cst, int S, int q0,
                                                     int nq) {
    const float* src[3] = {c.L0, c.ks, c.kd};
    float* dst = const_cast<float*>(c.cst);
    for (int sp = blockIdx.x * 256 + threadIdx.x; sp < S; sp += gridDim.x * 256) {
        const size_t base = (size_t)spring_cst[sp];
        for (int q = q0; q < q0 + nq; q++) dst[base + (size_t)q * c.N] = src[q][sp];
    }
}

hipError_t launch_scatter_cst(const DevCloth& c, const int32_t* spring_cst, int S, int q0, int nq,
                              hipStream_t st) {
    if (q0 < 0 || nq < 0 || q0 + nq > 3) return hipErrorInvalidValue;
    if (S <= 0 || nq == 0) return hipSuccess;
    const int grid = std::min((S + 255) / 256, 4096);
    hipLaunchKernelGGL(k_scatter_cst, dim3(grid), dim3(256), 0, st, c, spring_cst, S, q0, nq);
    return hipGetLastError();
}

hipError_t launch_cg_spmv(const DevCloth& c, const StepScalars& s, int k, hipStream_t st) {
    const dim3 grid(c.nt), block(kTileX * kTileY);
    if (c.stencil) return launch_k(1, k_cg_spmv<kTileX, kTileY, kStencil, true>, grid, block, st, c, s, k);
    if (c.wp <= 12) return launch_k(1, k_cg_spmv<kTileX, kTileY, 12, false>, grid, block, st, c, s, k);
    return launch_k(1, k_cg_spmv<kTileX, kTileY, kMaxPairWidth, false>, grid, block, st, c, s, k);
}

hipError_t launch_cg_axpy(const DevCloth& c, const StepScalars& s, int k, hipStream_t st) {
    return launch_k(2, k_cg_axpy<kTileX, kTileY>, dim3(c.nt), dim3(kTileX * kTileY), st, c, s, k);
}

hipError_t launch_cg_finish(const DevCloth& c, const StepScalars& s, hipStream_t st) {
    return launch_k(3, k_cg_finish, dim3(1), dim3(64), st, c, s);
}

int persistent_cg_grid(const DevCloth& c) {
    if (c.wp > 12) return 0;
    int dev = 0, coop = 0, cus = 0, per_cu = 0;
    if (!hip_ok(hipGetDevice(&dev)) || !hip_ok(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev)) ||
        !coop || !hip_ok(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) ||
        !hip_ok(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_cg_persistent<kTileX, kTileY, 12>, kTileX * kTileY,
                                                             0)))
        return 0;
    // Every block must own at least one tile: a block without one would not
    // see the stop decision and would wait at a barrier the others have
    // left.  Near-equal tile counts per block; a multiple of 8 blocks keeps
    // every tile a block serves on the block's XCD (tile_of_block).
    const int resident = per_cu * cus;
    if (resident < 1) return 0;
    const int per_block = (c.nt + resident - 1) / resident;
    int grid = (c.nt + per_block - 1) / per_block;
    if (grid >= 8) grid = grid / 8 * 8;
    return std::min(grid, c.nt);
}

// In a single iteration the blocks of a larger cloth do not win back what it
// takes to load what they keep and to exchange sums once (a step of one
// iteration, resident and with two launches: 512x512 53.7 and 48.4 us, 320x400
// 42.2 and 37.9, but 256x256 31.8 and 33.1; of two: 320x400 48.1 and 49.5).
static bool solves_resident(const DevCloth& c, const StepScalars& s) {
    return c.res_vt && s.max_it > (c.nt > kRowTiles ? 1 : 0) && !(s.flags & OC_FLAG_CG_SINGLE_REDUCTION);
}

bool assembles_rows(const DevCloth& c, const StepScalars& s) {
    return c.stencil_asm && c.res_vt == 1 && c.nt <= kRowTiles && solves_resident(c, s);
}

int resident_cg_tiles(const DevCloth& c) {
    int dev = 0, cus = 0;
    if (!c.stencil || c.nt > kResidentTiles || !hip_ok(hipGetDevice(&dev)) ||
        !hip_ok(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)))
        return 0;
    if (c.nt <= cus) return 1;
    return c.ntx * ((c.nty + 1) / 2) <= cus ? 2 : 0;
}

hipError_t launch_cg_resident(const DevCloth& c, const StepScalars& s, hipStream_t st, bool finish, int blocks) {
    const dim3 grid(blocks), block(kTileX * kTileY * c.res_vt);
    const int nb = resident_blocks(c.ntx, c.nty, c.res_vt);
    if (blocks < 1 || blocks > nb || s.max_it < 1) return hipErrorInvalidValue;
    if (c.res_vt == 1)
        return launch_k(1, k_cg_resident<kTileX, kTileY>, grid, block, st, c, s, nb, finish ? 1 : 0);
    if (c.res_vt == 2)
        return launch_k(1, k_cg_resident<kTileX, 2 * kTileY>, grid, block, st, c, s, nb, finish ? 1 : 0);
    return hipErrorInvalidValue;
}

hipError_t launch_cg(const DevCloth& c, const StepScalars& s, hipStream_t st, bool finish) {
    hipError_t e;
    if (solves_resident(c, s))
        return launch_cg_resident(c, s, st, finish, resident_blocks(c.ntx, c.nty, c.res_vt));
    if (c.persistent && s.max_it > 0 && !(s.flags & OC_FLAG_CG_SINGLE_REDUCTION)) {
        if (c.persistent > c.nt) return hipErrorInvalidValue;  // a block without a tile
        unsigned* bar = reinterpret_cast<unsigned*>(c.ctl + 6);
        hipLaunchKernelGGL(k_reset_barrier, dim3(1), dim3(64), 0, st, bar);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        DevCloth ca = c;
        StepScalars sa = s;
        void* args[] = {(void*)&ca, (void*)&sa, (void*)&bar};
        e = hipLaunchCooperativeKernel(
            reinterpret_cast<const void*>(k_cg_persistent<kTileX, kTileY, 12>), dim3(c.persistent),
            dim3(kTileX * kTileY), args, 0, st);
        if (e != hipSuccess) return e;
        return finish ? launch_cg_finish(c, s, st) : hipSuccess;
    }
    if (s.flags & OC_FLAG_CG_SINGLE_REDUCTION) {
        // the start: w0 = S A u0 and delta_0 (the first standard SpMV), then
        // one launch per iteration
        if (s.max_it > 0 && (e = launch_cg_spmv(c, s, 0, st)) != hipSuccess) return e;
        const dim3 grid(c.nt), block(kTileX * kTileY);
        for (int k = 0; k < s.max_it; k++) {
            if (c.stencil)
                e = launch_k(1, k_cg1<kTileX, kTileY, kStencil, true>, grid, block, st, c, s, k);
            else if (c.wp <= 12)
                e = launch_k(1, k_cg1<kTileX, kTileY, 12, false>, grid, block, st, c, s, k);
            else
                e = launch_k(1, k_cg1<kTileX, kTileY, kMaxPairWidth, false>, grid, block, st, c, s, k);
            if (e != hipSuccess) return e;
        }
        return finish ? launch_cg_finish(c, s, st) : hipSuccess;
    }
    for (int k = 0; k < s.max_it; k++) {
        if ((e = launch_cg_spmv(c, s, k, st)) != hipSuccess) return e;
        if ((e = launch_cg_axpy(c, s, k, st)) != hipSuccess) return e;
    }
    return finish ? launch_cg_finish(c, s, st) : hipSuccess;
}

hipError_t launch_update(const DevCloth& c, const StepScalars& s, hipStream_t st, bool finish, const oc_ellipsoid* e) {
    const dim3 grid((c.N + 255) / 256), block(256);
    const oc_ellipsoid el = e ? *e : oc_ellipsoid{};
    if (e)
        return finish ? launch_k(4, k_update<true, true>, grid, block, st, c, s, el)
                      : launch_k(4, k_update<false, true>, grid, block, st, c, s, el);
    return finish ? launch_k(4, k_update<true, false>, grid, block, st, c, s, el)
                  : launch_k(4, k_update<false, false>, grid, block, st, c, s, el);
}

}  // namespace oc
