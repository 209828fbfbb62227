// HIP kernels of the position-based-dynamics cloth step (gfx950, wave64),
// after OpenCloth_PositionBasedDynamics/.../main.cpp (PBD) with the triangle
// bending constraint (PBD:57).
//
//   pass_a    : gravity, global damping, V += (F dt) W; block partials of
//               m X, m V, m                         (PBD:601-631)
//   pass_b    : the first sums (one wave per scalar: block partials
//               lane-strided, 64-lane tree); R = X - Xcm; partials of
//               cross(R, m V) and m [R]x[R]x^T
//   tile      : one solver iteration: every colour in LDS, block by block;
//               the first predicts tmp_X (w = I^-1 L, centre-of-mass damping,
//               PBD:633-668), the last ends the step (PBD:670-678)
//   small     : whole steps of a cloth of up to 2048 particles, one workgroup
// and, for constraint graphs without a tiled plan,
//   pass_c    : the prediction
//   distance  : one colour of distance constraints  (PBD:680-701)
//   bending   : one colour of bending constraints   (PBD:703-731)
//   ground    : tmp_X.y < 0 -> 0                    (PBD:839-845)
//   integrate : V = (tmp_X - X)/dt, X = tmp_X       (PBD:670-678)
//
// The constraints of one colour share no particle, so a thread per
// constraint reproduces the sequential projection of that colour exactly;
// colours run in order.  The sums of the damping step use one fixed tree
// (64-lane shuffle trees, the 4 waves of a block in order, then the block
// partials lane-strided and one more tree), so results are deterministic
// and equal the CPU restatement with the same order bit for bit.
// Arithmetic follows the reference's GLM expression order (built with
// -ffp-contract=off).
#include <utility>

#include "oc_device.hpp"

namespace oc {

namespace {

using namespace dev;

constexpr int NB = kPbdBlock;
constexpr int NWB = NB / 64;

__device__ inline V3 cross3(V3 x, V3 y) {
    return {x.y * y.z - y.y * x.z, x.z * y.x - y.z * x.x, x.x * y.y - y.x * x.y};
}

// Velocity update of particle i (gravity, global damping, V += (F dt) W;
// PBD:601-631); returns the updated velocity.
__device__ __forceinline__ V3 external_force(const PbdScalars& s, V3 v, float wi) {
    const V3 F = wi > 0.0f ? V3{0.0f + s.gx, 0.0f + s.gy, 0.0f + s.gz} : V3{0.0f, 0.0f, 0.0f};
    v = {v.x * s.gd, v.y * s.gd, v.z * s.gd};
    return {v.x + (F.x * s.dt) * wi, v.y + (F.y * s.dt) * wi, v.z + (F.z * s.dt) * wi};
}
__device__ inline V3 external_velocity(const DevPbd& c, const PbdScalars& s, int i) {
    const V3 v = external_force(s, ld3(c.v, c.N, i), c.w[i]);
    st3(c.v, c.N, i, v);
    return v;
}

// Block partials of Q values per thread: wave trees, waves in order.
template <int Q>
__device__ inline void block_partials(const float (&t)[Q], float* part, int nblk, int first) {
    __shared__ float ws[Q][NWB];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const float s = wave_sum(t[q]);
        if (lane == 0) ws[q][wv] = s;
    }
    __syncthreads();
    if (threadIdx.x < Q) {
        const int q = threadIdx.x;
        float p = ws[q][0];
#pragma unroll
        for (int k = 1; k < NWB; k++) p = p + ws[q][k];
        part[(size_t)(first + q) * nblk + blockIdx.x] = p;
    }
}

// A particle's terms of the first sums: m X, m V, m (PBD:619-631).
__device__ __forceinline__ void sums_a(const PbdScalars& s, V3 x, V3 v, float (&t)[7]) {
    t[0] = x.x * s.mass;
    t[1] = x.y * s.mass;
    t[2] = x.z * s.mass;
    t[3] = v.x * s.mass;
    t[4] = v.y * s.mass;
    t[5] = v.z * s.mass;
    t[6] = s.mass;
}

// A particle's terms of the second: cross(R, m V) and m [R]x [R]x^T, which
// reduces exactly to these entries (xx yy zz xy xz yz).
__device__ __forceinline__ void sums_b(const PbdScalars& s, V3 xcm, V3 x, V3 v, float (&t)[9]) {
    const V3 R = {x.x - xcm.x, x.y - xcm.y, x.z - xcm.z};
    const V3 l = cross3(R, V3{s.mass * v.x, s.mass * v.y, s.mass * v.z});
    t[0] = l.x;
    t[1] = l.y;
    t[2] = l.z;
    t[3] = (R.y * R.y + R.z * R.z) * s.mass;
    t[4] = (R.x * R.x + R.z * R.z) * s.mass;
    t[5] = (R.x * R.x + R.y * R.y) * s.mass;
    t[6] = -(R.x * R.y) * s.mass;
    t[7] = -(R.x * R.z) * s.mass;
    t[8] = -(R.y * R.z) * s.mass;
}

__global__ __launch_bounds__(NB) void k_pbd_pass_a(DevPbd c, PbdScalars s) {
    const int i = blockIdx.x * NB + threadIdx.x;
    float t[7] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (i < c.N) {
        sums_a(s, ld3(c.x, c.N, i), external_velocity(c, s, i), t);
    }
    block_partials<7>(t, c.part, c.nblk, 0);
}

// One wave: lane-strided sum of nblk block partials, then a 64-lane tree
// (valid in lane 0).
__device__ __forceinline__ float sum_partials(const float* p, int nblk) {
    float s = 0.0f;
    for (int b = threadIdx.x & 63; b < nblk; b += 8 * 64) {
        float v[8];
#pragma unroll
        for (int q = 0; q < 8; q++) v[q] = p[min(b + 64 * q, nblk - 1)];
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (b + 64 * q < nblk) s += v[q];
    }
    return wave_sum(s);
}

__device__ inline V3 centre(const float* sums, int first) {
    return {sums[first] / sums[6], sums[first + 1] / sums[6], sums[first + 2] / sums[6]};
}

// The second sums' block partials.  Every workgroup finishes the first sums
// itself (7 waves, one sum each; the partials come from L2), which costs less
// than a launch of its own for them; workgroup 0 stores them for the
// prediction.  kPassB threads hold kPassB / NB reduction blocks.
constexpr int kPassB = 1024;
__global__ __launch_bounds__(kPassB) void k_pbd_pass_b(DevPbd c, PbdScalars s) {
    __shared__ float sums[8];
    __shared__ float ws[9][kPassB / 64];
    const int i = blockIdx.x * kPassB + threadIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    V3 x = {0.0f, 0.0f, 0.0f}, v = x;
    if (i < c.N) {
        x = ld3(c.x, c.N, i);
        v = ld3(c.v, c.N, i);
    }
    if (wv < 7) {
        const float q = sum_partials(c.part + (size_t)wv * c.nblk, c.nblk);
        if (lane == 0) {
            sums[wv] = q;
            if (blockIdx.x == 0) c.sums[wv] = q;
        }
    }
    __syncthreads();
    float t[9] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (i < c.N) sums_b(s, centre(sums, 0), x, v, t);
#pragma unroll
    for (int q = 0; q < 9; q++) {
        const float w = wave_sum(t[q]);
        if (lane == 0) ws[q][wv] = w;
    }
    __syncthreads();
    constexpr int G = kPassB / NB;
    if (threadIdx.x < 9 * G) {
        const int q = threadIdx.x / G, g = threadIdx.x % G, blk = blockIdx.x * G + g;
        if (blk < c.nblk) {
            float p = ws[q][g * NWB];
#pragma unroll
            for (int k = 1; k < NWB; k++) p = p + ws[q][g * NWB + k];
            c.part[(size_t)(7 + q) * c.nblk + blk] = p;
        }
    }
}

// w = I^-1 L (PBD:633-650) from the sums: I6 = I (xx yy zz xy xz yz), L =
// sum cross(R, m V).  I is inverted as glm::inverse does.
__device__ __forceinline__ V3 angular(const float* I6, const float* Lv) {
    const float xx = I6[0], yy = I6[1], zz = I6[2], xy = I6[3], xz = I6[4], yz = I6[5];
    const float M[3][3] = {{xx, xy, xz}, {xy, yy, yz}, {xz, yz, zz}};
    const float det = +M[0][0] * (M[1][1] * M[2][2] - M[2][1] * M[1][2]) -
                      M[1][0] * (M[0][1] * M[2][2] - M[2][1] * M[0][2]) +
                      M[2][0] * (M[0][1] * M[1][2] - M[1][1] * M[0][2]);
    float Inv[3][3];
    Inv[0][0] = +(M[1][1] * M[2][2] - M[2][1] * M[1][2]);
    Inv[1][0] = -(M[1][0] * M[2][2] - M[2][0] * M[1][2]);
    Inv[2][0] = +(M[1][0] * M[2][1] - M[2][0] * M[1][1]);
    Inv[0][1] = -(M[0][1] * M[2][2] - M[2][1] * M[0][2]);
    Inv[1][1] = +(M[0][0] * M[2][2] - M[2][0] * M[0][2]);
    Inv[2][1] = -(M[0][0] * M[2][1] - M[2][0] * M[0][1]);
    Inv[0][2] = +(M[0][1] * M[1][2] - M[1][1] * M[0][2]);
    Inv[1][2] = -(M[0][0] * M[1][2] - M[1][0] * M[0][2]);
    Inv[2][2] = +(M[0][0] * M[1][1] - M[1][0] * M[0][1]);
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++) Inv[a][b] = Inv[a][b] / det;
    const float L[3] = {Lv[0], Lv[1], Lv[2]};
    V3 w;
    w.x = Inv[0][0] * L[0] + Inv[1][0] * L[1] + Inv[2][0] * L[2];
    w.y = Inv[0][1] * L[0] + Inv[1][1] * L[1] + Inv[2][1] * L[2];
    w.z = Inv[0][2] * L[0] + Inv[1][2] * L[1] + Inv[2][2] * L[2];
    return w;
}

// Centre-of-mass damping (v updated) and prediction of a particle (PBD:651-668).
__device__ __forceinline__ V3 damp_predict(const PbdScalars& s, V3 w, V3 xcm, V3 vcm, V3 x, V3& v, float wi) {
    const V3 R = {x.x - xcm.x, x.y - xcm.y, x.z - xcm.z};
    const V3 wr = cross3(w, R);
    const V3 del = {(vcm.x + wr.x) - v.x, (vcm.y + wr.y) - v.y, (vcm.z + wr.z) - v.z};
    v = {v.x + s.kdamp * del.x, v.y + s.kdamp * del.y, v.z + s.kdamp * del.z};
    return wi <= 0.0f ? x : V3{x.x + v.x * s.dt, x.y + v.y * s.dt, x.z + v.z * s.dt};
}

// What the prediction needs of the sums, by one thread: w, the centres.
struct PbdMotion {
    V3 w, xcm, vcm;
};
__device__ __forceinline__ PbdMotion motion_of(const float* S) {
    // I = identity + sum (symmetric, column-major m[c][r])
    const float I6[6] = {1.0f + S[10], 1.0f + S[11], 1.0f + S[12], 0.0f + S[13], 0.0f + S[14], 0.0f + S[15]};
    return {angular(I6, S + 7), centre(S, 0), centre(S, 3)};
}

// The prediction per particle, for the per-colour form (the second sums
// finished by every workgroup, as in pass b).
__global__ __launch_bounds__(kPassB) void k_pbd_pass_c(DevPbd c, PbdScalars s) {
    __shared__ float S[kPbdSums];
    __shared__ PbdMotion mo;
    const int i = blockIdx.x * kPassB + threadIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (wv < 9) {
        const float q = sum_partials(c.part + (size_t)(7 + wv) * c.nblk, c.nblk);
        if (lane == 0) S[7 + wv] = q;
    } else if (wv == 9 && lane < 7) {
        S[lane] = c.sums[lane];
    }
    __syncthreads();
    if (threadIdx.x == 0) mo = motion_of(S);
    __syncthreads();
    if (i >= c.N) return;
    V3 v = ld3(c.v, c.N, i);
    st3(c.t, c.N, i, damp_predict(s, mo.w, mo.xcm, mo.vcm, ld3(c.x, c.N, i), v, c.w[i]));
}

// The prediction with the reference's sequential sums (list order): one
// workgroup; thread 0 adds the centre-of-mass sums in particle order and
// accumulates I onto the identity, as PBD:612-650 does; every particle's
// update runs in parallel.
constexpr int kSeqThreads = 1024;
__global__ __launch_bounds__(kSeqThreads) void k_pbd_predict_seq(DevPbd c, PbdScalars s) {
    __shared__ float sx[3], sv[3], sI[6], sL[3];
    for (int i = threadIdx.x; i < c.N; i += kSeqThreads) external_velocity(c, s, i);
    __syncthreads();
    if (threadIdx.x == 0) {
        float xs[3] = {0.0f, 0.0f, 0.0f}, vs[3] = {0.0f, 0.0f, 0.0f}, ms = 0.0f;
        for (int i = 0; i < c.N; i++) {
            const V3 x = ld3(c.x, c.N, i), v = ld3(c.v, c.N, i);
            xs[0] += x.x * s.mass;
            xs[1] += x.y * s.mass;
            xs[2] += x.z * s.mass;
            vs[0] += v.x * s.mass;
            vs[1] += v.y * s.mass;
            vs[2] += v.z * s.mass;
            ms += s.mass;
        }
        const V3 xcm = {xs[0] / ms, xs[1] / ms, xs[2] / ms};
        float L[3] = {0.0f, 0.0f, 0.0f}, I6[6] = {1.0f, 1.0f, 1.0f, 0.0f, 0.0f, 0.0f};
        for (int i = 0; i < c.N; i++) {
            const V3 x = ld3(c.x, c.N, i), v = ld3(c.v, c.N, i);
            const V3 R = {x.x - xcm.x, x.y - xcm.y, x.z - xcm.z};
            const V3 l = cross3(R, V3{s.mass * v.x, s.mass * v.y, s.mass * v.z});
            L[0] += l.x;
            L[1] += l.y;
            L[2] += l.z;
            I6[0] += (R.y * R.y + R.z * R.z) * s.mass;
            I6[1] += (R.x * R.x + R.z * R.z) * s.mass;
            I6[2] += (R.x * R.x + R.y * R.y) * s.mass;
            I6[3] += -(R.x * R.y) * s.mass;
            I6[4] += -(R.x * R.z) * s.mass;
            I6[5] += -(R.y * R.z) * s.mass;
        }
        for (int k = 0; k < 3; k++) {
            sx[k] = k == 0 ? xcm.x : k == 1 ? xcm.y : xcm.z;
            sv[k] = vs[k] / ms;
            sL[k] = L[k];
        }
        for (int k = 0; k < 6; k++) sI[k] = I6[k];
    }
    __syncthreads();
    const V3 w = angular(sI, sL);
    for (int i = threadIdx.x; i < c.N; i += kSeqThreads) {
        V3 v = ld3(c.v, c.N, i);
        st3(c.t, c.N, i,
            damp_predict(s, w, V3{sx[0], sx[1], sx[2]}, V3{sv[0], sv[1], sv[2]}, ld3(c.x, c.N, i), v, c.w[i]));
    }
}

// UpdateDistanceConstraint (PBD:680-701): the move dP of the first particle
// per unit of inverse mass (the second moves the other way); false for none.
__device__ __forceinline__ bool distance_move(const PbdScalars& s, V3 ta, V3 tb, float w1, float w2, float rest,
                                              float kp, V3& dP) {
    const V3 dir = {ta.x - tb.x, ta.y - tb.y, ta.z - tb.z};
    const float len = sqrtf(dir.x * dir.x + dir.y * dir.y + dir.z * dir.z);
    if (len <= 0.0000001f) return false;
    const float inv_mass = w1 + w2;
    if (inv_mass <= 0.0000001f) return false;
    float inv = s.inv_2w;  // two free particles
    if (w1 != s.w || w2 != s.w) inv = 1.0f / inv_mass;
    const float sc = inv * (len - rest);
    dP = {(sc * (dir.x / len)) * kp, (sc * (dir.y / len)) * kp, (sc * (dir.z / len)) * kp};
    return true;
}

__device__ inline V3 minus_scaled(V3 t, V3 d, float w) { return {t.x - d.x * w, t.y - d.y * w, t.z - d.z * w}; }
__device__ inline V3 plus_scaled(V3 t, V3 d, float w) { return {t.x + d.x * w, t.y + d.y * w, t.z + d.z * w}; }
__device__ inline V3 plus_times(V3 t, float s, V3 f) { return {t.x + s * f.x, t.y + s * f.y, t.z + s * f.z}; }

// Stored constraint k.
__device__ inline void project_distance(const DevPbd& c, const PbdScalars& s, int k) {
    const int a = c.d_p1[k], b = c.d_p2[k];
    const float w1 = c.w[a], w2 = c.w[b];
    const V3 ta = ld3(c.t, c.N, a), tb = ld3(c.t, c.N, b);
    V3 dP;
    if (!distance_move(s, ta, tb, w1, w2, c.d_rest[k], c.d_kp[k], dP)) return;
    if (w1 > 0.0f) st3(c.t, c.N, a, minus_scaled(ta, dP, w1));
    if (w2 > 0.0f) st3(c.t, c.N, b, plus_scaled(tb, dP, w2));
}

__global__ __launch_bounds__(256) void k_pbd_distance(DevPbd c, PbdScalars s, int first, int count) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < count) project_distance(c, s, first + j);
}

// UpdateBendingConstraint (PBD:703-731): the moves of the three particles,
// f times m[0..2].
__device__ __forceinline__ void bending_move(const PbdScalars& s, V3 ta, V3 tb, V3 td, float wa, float wb, float wd, float wsum,
                                    float rest, float kp, V3& f, float (&m)[3]) {
    const V3 ctr = {0.3333f * ((ta.x + tb.x) + td.x), 0.3333f * ((ta.y + tb.y) + td.y),
                    0.3333f * ((ta.z + tb.z) + td.z)};
    const V3 dc = {td.x - ctr.x, td.y - ctr.y, td.z - ctr.z};
    const float dist = sqrtf(dc.x * dc.x + dc.y * dc.y + dc.z * dc.z);
    const float diff = 1.0f - ((s.global_k + rest) / dist);
    f = {dc.x * diff, dc.y * diff, dc.z * diff};
    float ra = s.bend_2w, rb = s.bend_2w, rd = s.bend_4w;  // three free particles
    if (wa != s.w || wb != s.w || wd != s.w) {
        ra = (2.0f * wa) / wsum;
        rb = (2.0f * wb) / wsum;
        rd = (4.0f * wd) / wsum;
    }
    m[0] = kp * ra;
    m[1] = kp * rb;
    m[2] = -kp * rd;
}

// Stored constraint k.
__device__ inline void project_bending(const DevPbd& c, const PbdScalars& s, int k) {
    const int a = c.b_p1[k], b = c.b_p2[k], d = c.b_p3[k];
    const float wa = c.w[a], wb = c.w[b], wd = c.w[d];
    const V3 ta = ld3(c.t, c.N, a), tb = ld3(c.t, c.N, b), td = ld3(c.t, c.N, d);
    V3 f;
    float m[3];
    bending_move(s, ta, tb, td, wa, wb, wd, c.b_w[k], c.b_rest[k], c.b_kp[k], f, m);
    if (wa > 0.0f) st3(c.t, c.N, a, plus_times(ta, m[0], f));
    if (wb > 0.0f) st3(c.t, c.N, b, plus_times(tb, m[1], f));
    if (wd > 0.0f) st3(c.t, c.N, d, plus_times(td, m[2], f));
}

__global__ __launch_bounds__(256) void k_pbd_bending(DevPbd c, PbdScalars s, int first, int count) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < count) project_bending(c, s, first + j);
}

// The list-order schedule in one workgroup.  The constraints of a level
// touch disjoint particles and every earlier constraint sharing a particle
// with one of them sits in an earlier level, so projecting the levels in
// order, a level's constraints in parallel, gives the sequential list order's
// results (UpdateInternalConstraints, PBD:876-889).  The workgroup barrier
// after each level orders the global memory accesses of the one workgroup.
constexpr int kLevelThreads = 1024;
__global__ __launch_bounds__(kLevelThreads) void k_pbd_levels(DevPbd c, PbdScalars s, int iterations,
                                                             int ground) {
    for (int it = 0; it < iterations; it++) {
        for (int L = 0; L < c.nd_lv; L++) {
            const int first = c.d_lv[L], last = c.d_lv[L + 1];
            for (int k = first + (int)threadIdx.x; k < last; k += kLevelThreads) project_distance(c, s, k);
            __syncthreads();
        }
        for (int L = 0; L < c.nb_lv; L++) {
            const int first = c.b_lv[L], last = c.b_lv[L + 1];
            for (int k = first + (int)threadIdx.x; k < last; k += kLevelThreads) project_bending(c, s, k);
            __syncthreads();
        }
        if (ground) {  // GroundCollision (PBD:839-845)
            for (int i = threadIdx.x; i < c.N; i += kLevelThreads) {
                float* ty = c.t + c.N + i;
                if (*ty < 0.0f) *ty = 0.0f;
            }
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(256) void k_pbd_ground(DevPbd c) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= c.N) return;
    float* ty = c.t + c.N + i;
    if (*ty < 0.0f) *ty = 0.0f;
}

__global__ __launch_bounds__(256) void k_pbd_integrate(DevPbd c, PbdScalars s) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= c.N) return;
    const V3 t = ld3(c.t, c.N, i), x = ld3(c.x, c.N, i);
    st3(c.v, c.N, i, V3{(t.x - x.x) * s.inv_dt, (t.y - x.y) * s.inv_dt, (t.z - x.z) * s.inv_dt});
    st3(c.x, c.N, i, t);
}

// ---------------------------------------------------------------------------
// tiled solver: a workgroup projects its closure (pbd_plan.cpp) in LDS
// ---------------------------------------------------------------------------
// One launch per colour took 4.5 us and more at any size, launch and latency
// (14 colours per solver iteration on the reference's lists).  Here a solver
// iteration is one launch: a workgroup loads its owned particles and their
// surroundings, projects every colour in LDS with a barrier in between, and
// writes the owned particles.  At 1024 owned particles a workgroup of the
// 512x512 grid holds 2311 particles and projects 1.95 times its share of the
// distance and 1.28 times its share of the bending constraints; larger blocks
// repeat less but leave CUs idle.  A particle (position and inverse mass, 16
// bytes) moves in one LDS instruction; records are loaded a few colours
// ahead.  What bounds it is the chain through a colour (LDS read, square
// root, divisions, LDS write, barrier): about 1300 cycles each with one wave
// per SIMD, 1500 with four.  Time per step before and now: 64x64 139 -> 37
// us, 256x256 140 -> 43, 512x512 181 -> 49 (two tile launches of 21, sums 5
// and 5).

// All colours of one solver iteration over the workgroup's particles tp.  A
// thread's first ROUNDS records of a colour are loaded kAhead colours before
// they are projected, by unconditional loads (a thread without a constraint
// loads some other record), so that the compiler can wait for exactly the
// loads it needs.  KP: the constraints have their own k'.
constexpr int kAhead = 3;
template <int NT, int ROUNDS, bool KP>
__device__ __forceinline__ void project_colours(const DevPbd& c, const PbdScalars& s, const int* cptr, float4* tp) {
    const int nd = c.nd_col, ncol = nd + c.nb_col, tid = threadIdx.x, end = c.n_rec - 1;
    const float d_all = c.d_kp_all, b_all = c.b_kp_all;
    struct Item {
        PbdRecord r;
        float kp;
    };
    auto fetch = [&](int k) {
        const int i = min(k, end);
        Item e;
        e.r = c.t_rec[i];
        e.kp = KP ? c.t_kp[i] : 0.0f;
        return e;
    };
    auto project = [&](int col, const Item& e) {
        const unsigned A = e.r.ab & 0xFFFFu, B = e.r.ab >> 16;
        const float4 a = tp[A], b = tp[B];
        const V3 ta = {a.x, a.y, a.z}, tb = {b.x, b.y, b.z};
        auto put = [&](unsigned p, V3 t, float w) { tp[p] = make_float4(t.x, t.y, t.z, w); };
        if (col < nd) {
            V3 dP;
            if (distance_move(s, ta, tb, a.w, b.w, e.r.rest, KP ? e.kp : d_all, dP)) {
                if (a.w > 0.0f) put(A, minus_scaled(ta, dP, a.w), a.w);
                if (b.w > 0.0f) put(B, plus_scaled(tb, dP, b.w), b.w);
            }
        } else {
            const unsigned D = e.r.c;
            const float4 d = tp[D];
            const V3 td = {d.x, d.y, d.z};
            V3 f;
            float m[3];
            // (the sum of inverse masses as oc_pbd_create forms it)
            const float wsum = a.w + b.w + 2.0f * d.w;
            bending_move(s, ta, tb, td, a.w, b.w, d.w, wsum, e.r.rest, KP ? e.kp : b_all, f, m);
            if (a.w > 0.0f) put(A, plus_times(ta, m[0], f), a.w);
            if (b.w > 0.0f) put(B, plus_times(tb, m[1], f), b.w);
            if (d.w > 0.0f) put(D, plus_times(td, m[2], f), d.w);
        }
    };
    Item nxt[kAhead][ROUNDS];
    auto refill = [&](Item (&n)[ROUNDS], int lo) {
#pragma unroll
        for (int q = 0; q < ROUNDS; q++) n[q] = fetch(lo + tid + q * NT);
    };
#pragma unroll
    for (int u = 0; u < kAhead; u++) refill(nxt[u], cptr[min(u, ncol)]);
    for (int col = 0; col < ncol; col += kAhead)
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            if (col + u >= ncol) break;
            const int lo = cptr[col + u], hi = cptr[col + u + 1];
            Item r[ROUNDS];
#pragma unroll
            for (int q = 0; q < ROUNDS; q++) r[q] = nxt[u][q];
            refill(nxt[u], cptr[min(col + u + kAhead, ncol)]);
#pragma unroll
            for (int q = 0; q < ROUNDS; q++)
                if (lo + tid + q * NT < hi) project(col + u, r[q]);
            for (int k = lo + tid + ROUNDS * NT; k < hi; k += NT) project(col + u, fetch(k));
            __syncthreads();
        }
}

constexpr int kTileThreads = 1024;
constexpr int kMaxColours = 128;  // of both families

// One solver iteration.  FIRST: the particles are predicted from x and v
// (the second sums finished here, as in pass c); else they come from t.
// LAST: collider, velocities, results to x and v (in place: it reads x of its
// owned particles only); else to t2.
template <bool FIRST, bool LAST, bool KP>
__global__ __launch_bounds__(kTileThreads) void k_pbd_tile(DevPbd c, PbdScalars s, oc_ellipsoid e, int has_e) {
    static_assert(!(FIRST && LAST), "every block reads its surroundings' x and v before they change");
    extern __shared__ float4 tp[];
    __shared__ int cptr[kMaxColours + 1];
    __shared__ float S[kPbdSums];
    __shared__ PbdMotion mo;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, ncol = c.nd_col + c.nb_col;
    // XCD x takes a run of neighbouring blocks, whose surroundings overlap
    const int nb = c.nb, xb = blockIdx.x & 7, xq = nb >> 3, xr = nb & 7;
    const int blk = xb * xq + min(xb, xr) + ((int)blockIdx.x >> 3);
    const int off = c.t_off[blk], nl = c.t_off[blk + 1] - off, nown = c.t_own[blk];
    if (tid <= ncol) cptr[tid] = c.t_cptr[blk * (ncol + 1) + tid];
    if constexpr (FIRST) {
        if (wv < 9) {
            const float q = sum_partials(c.part + (size_t)(7 + wv) * c.nblk, c.nblk);
            if (lane == 0) S[7 + wv] = q;
        } else if (wv == 9 && lane < 7) {
            S[lane] = c.sums[lane];
        }
        __syncthreads();
        if (tid == 0) mo = motion_of(S);
        __syncthreads();
    }
    for (int k = tid; k < nl; k += kTileThreads) {
        const int i = c.t_ids[off + k];
        const float w = c.w[i];
        V3 t;
        if constexpr (FIRST) {
            V3 v = ld3(c.v, c.N, i);
            t = damp_predict(s, mo.w, mo.xcm, mo.vcm, ld3(c.x, c.N, i), v, w);
        } else {
            t = ld3(c.t, c.N, i);
        }
        tp[k] = make_float4(t.x, t.y, t.z, w);
    }
    __syncthreads();
    project_colours<kTileThreads, 2, KP>(c, s, cptr, tp);
    for (int k = tid; k < nown; k += kTileThreads) {
        const int i = c.t_ids[off + k];
        V3 t = {tp[k].x, tp[k].y, tp[k].z};
        if ((s.flags & OC_FLAG_GROUND_CLAMP) && t.y < 0.0f) t.y = 0.0f;  // GroundCollision (PBD:839-845)
        if constexpr (LAST) {
            bool inside;
            if (has_e) t = ellipsoid_push(e, t, inside);
            const V3 x = ld3(c.x, c.N, i);
            st3(c.v, c.N, i, V3{(t.x - x.x) * s.inv_dt, (t.y - x.y) * s.inv_dt, (t.z - x.z) * s.inv_dt});
            st3(c.x, c.N, i, t);
        } else {
            st3(c.t2, c.N, i, t);
        }
    }
}

// Whole steps of a cloth of at most PT * NT particles by one workgroup: sums,
// prediction, every solver iteration, collider and velocities, with x and v
// in registers and the predicted positions in LDS.  The sums keep the block
// and lane trees of the passes above (virtual blocks of NB particles).  A
// 21x21 step took 132 us in 35 launches and takes 17 here, 83% of it in the
// colours' chains.
template <int NT, int PT, bool KP>
__global__ __launch_bounds__(NT) void k_pbd_small(DevPbd c, PbdScalars s, int nsteps, int iterations, oc_ellipsoid e,
                                                  int has_e) {
    extern __shared__ float4 tp[];
    constexpr int NV = (NT * PT + NB - 1) / NB;  // virtual reduction blocks
    static_assert(NT / 64 >= 8 && NV <= 64, "a wave per sum (two rounds for nine), a lane per block");
    __shared__ int cptr[kMaxColours + 1];
    __shared__ float ws[9][NV * NWB];
    __shared__ float S[kPbdSums];
    __shared__ PbdMotion mo;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, N = c.N;
    if (tid <= c.nd_col + c.nb_col) cptr[tid] = c.t_cptr[tid];
    V3 x[PT], v[PT];
    float w[PT];
#pragma unroll
    for (int j = 0; j < PT; j++) {
        const int i = tid + j * NT;
        x[j] = v[j] = V3{0.0f, 0.0f, 0.0f};
        w[j] = 0.0f;
        if (i < N) {
            x[j] = ld3(c.x, N, i);
            v[j] = ld3(c.v, N, i);
            w[j] = c.w[i];
        }
    }
    // the sums in ws (wave sums by virtual wave) finished into S[first ...]
    auto finish = [&](int first, int count) {
        __syncthreads();
        for (int q = wv; q < count; q += NT / 64) {
            float p = 0.0f;
            if (lane < c.nblk) {
                p = ws[q][lane * NWB];
#pragma unroll
                for (int k = 1; k < NWB; k++) p = p + ws[q][lane * NWB + k];
            }
            p = wave_sum(0.0f + p);
            if (lane == 0) S[first + q] = p;
        }
        __syncthreads();
    };
    for (int n = 0; n < nsteps; n++) {
#pragma unroll
        for (int j = 0; j < PT; j++) {
            float t[7] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            if (tid + j * NT < N) {
                v[j] = external_force(s, v[j], w[j]);
                sums_a(s, x[j], v[j], t);
            }
#pragma unroll
            for (int q = 0; q < 7; q++) {
                const float p = wave_sum(t[q]);
                if (lane == 0) ws[q][j * (NT / 64) + wv] = p;
            }
        }
        finish(0, 7);
        const V3 xcm = centre(S, 0);
#pragma unroll
        for (int j = 0; j < PT; j++) {
            float t[9] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
            if (tid + j * NT < N) sums_b(s, xcm, x[j], v[j], t);
#pragma unroll
            for (int q = 0; q < 9; q++) {
                const float p = wave_sum(t[q]);
                if (lane == 0) ws[q][j * (NT / 64) + wv] = p;
            }
        }
        finish(7, 9);
        if (tid == 0) mo = motion_of(S);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < PT; j++)
            if (tid + j * NT < N) {
                const V3 t = damp_predict(s, mo.w, mo.xcm, mo.vcm, x[j], v[j], w[j]);
                tp[tid + j * NT] = make_float4(t.x, t.y, t.z, w[j]);
            }
        __syncthreads();
        for (int it = 0; it < iterations; it++) {
            project_colours<NT, 1, KP>(c, s, cptr, tp);
            if (s.flags & OC_FLAG_GROUND_CLAMP) {
                for (int i = tid; i < N; i += NT)
                    if (tp[i].y < 0.0f) tp[i].y = 0.0f;
                __syncthreads();
            }
        }
#pragma unroll
        for (int j = 0; j < PT; j++)
            if (tid + j * NT < N) {
                V3 t = {tp[tid + j * NT].x, tp[tid + j * NT].y, tp[tid + j * NT].z};
                bool inside;
                if (has_e) t = ellipsoid_push(e, t, inside);
                v[j] = {(t.x - x[j].x) * s.inv_dt, (t.y - x[j].y) * s.inv_dt, (t.z - x[j].z) * s.inv_dt};
                x[j] = t;
            }
    }
#pragma unroll
    for (int j = 0; j < PT; j++)
        if (tid + j * NT < N) {
            st3(c.x, N, tid + j * NT, x[j]);
            st3(c.v, N, tid + j * NT, v[j]);
        }
}

}  // namespace

template <bool KP>
static hipError_t launch_small(const DevPbd& c, const PbdScalars& s, int nsteps, int iterations, const oc_ellipsoid* e,
                               hipStream_t st) {
    const oc_ellipsoid el = e ? *e : oc_ellipsoid{};
    const int has_e = e != nullptr;
    const size_t lds = sizeof(float4) * (size_t)c.N;
    if (c.N <= 512)
        hipLaunchKernelGGL((k_pbd_small<512, 1, KP>), dim3(1), dim3(512), lds, st, c, s, nsteps, iterations, el, has_e);
    else if (c.N <= 1024)
        hipLaunchKernelGGL((k_pbd_small<1024, 1, KP>), dim3(1), dim3(1024), lds, st, c, s, nsteps, iterations, el, has_e);
    else
        hipLaunchKernelGGL((k_pbd_small<1024, 2, KP>), dim3(1), dim3(1024), lds, st, c, s, nsteps, iterations, el, has_e);
    return hipGetLastError();
}

hipError_t launch_pbd_small(const DevPbd& c, const PbdScalars& s, int nsteps, int iterations, const oc_ellipsoid* e,
                            hipStream_t st) {
    static_assert(kPbdSmall == 2 * 1024, "the largest instance");
    if (c.nb != 1 || c.N > kPbdSmall || c.nd_col + c.nb_col > kMaxColours) return hipErrorInvalidValue;
    return c.t_kp ? launch_small<true>(c, s, nsteps, iterations, e, st)
                  : launch_small<false>(c, s, nsteps, iterations, e, st);
}

// The sums of a step: the first sums' partials (v updated), the second's.
static void launch_sums(const DevPbd& c, const PbdScalars& s, hipStream_t st) {
    hipLaunchKernelGGL(k_pbd_pass_a, dim3(c.nblk), dim3(NB), 0, st, c, s);
    hipLaunchKernelGGL(k_pbd_pass_b, dim3((c.N + kPassB - 1) / kPassB), dim3(kPassB), 0, st, c, s);
}

template <bool FIRST, bool LAST>
static void launch_tile(const DevPbd& c, const PbdScalars& s, const oc_ellipsoid* e, hipStream_t st) {
    const oc_ellipsoid el = e ? *e : oc_ellipsoid{};
    const size_t lds = sizeof(float4) * (size_t)c.max_local;
    if (c.t_kp)
        hipLaunchKernelGGL((k_pbd_tile<FIRST, LAST, true>), dim3(c.nb), dim3(kTileThreads), lds, st, c, s, el, e != nullptr);
    else
        hipLaunchKernelGGL((k_pbd_tile<FIRST, LAST, false>), dim3(c.nb), dim3(kTileThreads), lds, st, c, s, el, e != nullptr);
}

hipError_t launch_pbd_tiled(const DevPbd& c, const PbdScalars& s, int iterations, const oc_ellipsoid* e,
                            hipStream_t st) {
    if (c.nb < 2 || iterations < 1 || c.nd_col + c.nb_col > kMaxColours) return hipErrorInvalidValue;
    launch_sums(c, s, st);
    DevPbd d = c;
    for (int it = 0; it < iterations; it++) {
        if (it == 0)
            launch_tile<true, false>(d, s, e, st);
        else if (it + 1 == iterations)
            launch_tile<false, true>(d, s, e, st);
        else
            launch_tile<false, false>(d, s, e, st);
        std::swap(d.t, d.t2);
    }
    if (iterations > 1) return hipGetLastError();
    if (e) {
        const hipError_t r = launch_ellipsoid(d.t, d.v, d.N, *e, 0, st);
        if (r != hipSuccess) return r;
    }
    return launch_pbd_integrate(d, s, st);
}

hipError_t launch_pbd_predict(const DevPbd& c, const PbdScalars& s, hipStream_t st) {
    launch_sums(c, s, st);
    hipLaunchKernelGGL(k_pbd_pass_c, dim3((c.N + kPassB - 1) / kPassB), dim3(kPassB), 0, st, c, s);
    return hipGetLastError();
}

hipError_t launch_pbd_distance(const DevPbd& c, const PbdScalars& s, int first, int count, hipStream_t st) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pbd_distance, dim3((count + 255) / 256), dim3(256), 0, st, c, s, first, count);
    return hipGetLastError();
}

hipError_t launch_pbd_bending(const DevPbd& c, const PbdScalars& s, int first, int count,
                              hipStream_t st) {
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pbd_bending, dim3((count + 255) / 256), dim3(256), 0, st, c, s, first,
                       count);
    return hipGetLastError();
}

hipError_t launch_pbd_predict_seq(const DevPbd& c, const PbdScalars& s, hipStream_t st) {
    hipLaunchKernelGGL(k_pbd_predict_seq, dim3(1), dim3(kSeqThreads), 0, st, c, s);
    return hipGetLastError();
}

hipError_t launch_pbd_levels(const DevPbd& c, const PbdScalars& s, int iterations, int ground,
                             hipStream_t st) {
    hipLaunchKernelGGL(k_pbd_levels, dim3(1), dim3(kLevelThreads), 0, st, c, s, iterations, ground);
    return hipGetLastError();
}

hipError_t launch_pbd_ground(const DevPbd& c, hipStream_t st) {
    hipLaunchKernelGGL(k_pbd_ground, dim3((c.N + 255) / 256), dim3(256), 0, st, c);
    return hipGetLastError();
}

hipError_t launch_pbd_integrate(const DevPbd& c, const PbdScalars& s, hipStream_t st) {
    hipLaunchKernelGGL(k_pbd_integrate, dim3((c.N + 255) / 256), dim3(256), 0, st, c, s);
    return hipGetLastError();
}

}  // namespace oc
