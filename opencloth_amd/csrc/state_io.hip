// State transfers: host arrays of vertices (xyz or xyzw, the caller's layout)
// to and from the SoA planes on the device.  A kernel packs the planes
// straight into pinned host memory (or unpacks from it), so that the layout
// change costs no pass over memory of its own, and the host only copies
// between the pinned slots and the caller's arrays.
//
// What bounds it: launch and synchronisation for small states (16 us at 441
// vertices, 48 with a copy and a host transpose per array), the host link for
// large ones (56 GB/s when device memory is copied to pinned memory; 24.6 MB
// of 1023x1001 vertices in 640 us, 5.3 ms before) and the page faults of the
// caller's fresh arrays.  Up to one slot both arrays of a state go in a
// single launch with one synchronisation, and one array alone by a copy where
// that is quicker; beyond it, the host copy of one
// slot overlaps the transfer of the next, and larger transfers have more host
// threads with slots of their own.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "oc_internal.hpp"

namespace oc {

namespace {

constexpr size_t kSlot = 21846 * 48;          // bytes: about 1 MiB, whole vertices of 3 and of 4 floats
// Bytes of a transfer for each host thread: the 6.3 MB state of 262144
// vertices into fresh arrays takes 1350 us with one thread, 810 with four;
// with arrays whose pages are there threads gain and lose nothing.
constexpr size_t kPerThread = 2u << 20;
constexpr int kThreads = 4;
// One array of xyz of more than this, up to a slot, is transposed by the host
// and copied: above 16 KiB the runtime's copy takes 9 us with its
// synchronisation, where a launch that packs takes 14 (one array of 4096
// vertices: 11 us, packed 16; of 16384: 17 and 21; below, 12 to 14 for the
// copy alone).  Two arrays would be two copies.
constexpr size_t kCopy = 16384;

int threads_of(size_t total) { return (int)std::min<size_t>(kThreads, 1 + total / kPerThread); }

// m vertices, of planes p (stride n) and the fourth components w, as quads
// of floats.
struct Part {
    float* p;
    float* w;
    size_t n;
    unsigned m, quads;
};

template <int C>
__global__ __launch_bounds__(256) void k_pack(Part a, Part b, float4* out) {
    unsigned t = blockIdx.x * 256 + threadIdx.x;
    if (t >= a.quads + b.quads) return;
    float4* const dst = out + t;
    Part s = a;
    if (t >= a.quads) {
        s = b;
        t -= a.quads;
    }
    float4 q;
    if constexpr (C == 4) {
        q = make_float4(s.p[t], s.p[s.n + t], s.p[2 * s.n + t], s.w[t]);
    } else {
        float v[4];
#pragma unroll
        for (unsigned j = 0; j < 4; j++) {
            const unsigned k = 4 * t + j, i = k / 3;
            v[j] = i < s.m ? s.p[(k - 3 * i) * s.n + i] : 0.0f;
        }
        q = make_float4(v[0], v[1], v[2], v[3]);
    }
    *dst = q;
}

template <int C>
__global__ __launch_bounds__(256) void k_unpack(Part a, Part b, const float4* in) {
    unsigned t = blockIdx.x * 256 + threadIdx.x;
    if (t >= a.quads + b.quads) return;
    const float4 q = in[t];
    Part s = a;
    if (t >= a.quads) {
        s = b;
        t -= a.quads;
    }
    if constexpr (C == 4) {
        s.p[t] = q.x;
        s.p[s.n + t] = q.y;
        s.p[2 * s.n + t] = q.z;
        s.w[t] = q.w;
    } else {
        const float v[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (unsigned j = 0; j < 4; j++) {
            const unsigned k = 4 * t + j, i = k / 3;
            if (i < s.m) s.p[(k - 3 * i) * s.n + i] = v[j];
        }
    }
}

unsigned quads_of(size_t m, int comps) { return (unsigned)((m * comps + 3) / 4); }

hipError_t launch(bool read, int comps, const Part& a, const Part& b, char* slot, hipStream_t st) {
    const unsigned q = a.quads + b.quads;
    const dim3 g((q + 255) / 256), t(256);
    if (q == 0) return hipSuccess;
    if (read && comps == 4)
        hipLaunchKernelGGL(k_pack<4>, g, t, 0, st, a, b, (float4*)slot);
    else if (read)
        hipLaunchKernelGGL(k_pack<3>, g, t, 0, st, a, b, (float4*)slot);
    else if (comps == 4)
        hipLaunchKernelGGL(k_unpack<4>, g, t, 0, st, a, b, (const float4*)slot);
    else
        hipLaunchKernelGGL(k_unpack<3>, g, t, 0, st, a, b, (const float4*)slot);
    return hipGetLastError();
}

Part part_of(const IoArray& a, size_t v0, size_t m) {
    return {a.planes + v0, a.w ? a.w + v0 : nullptr, a.n, (unsigned)m, quads_of(m, a.comps())};
}

}  // namespace

StateIo::~StateIo() {
    for (hipEvent_t e : ev_)
        if (e) (void)hipEventDestroy(e);
    if (pinned_) (void)hipHostFree(pinned_);
}

// The slots of a transfer of total bytes, kept for later calls: what it needs
// up to one slot, beyond that two for each of its threads.
hipError_t StateIo::reserve(size_t total) {
    const int slots = total <= kSlot ? 1 : 2 * threads_of(total);
    const size_t need = total <= kSlot ? (total + 4095) / 4096 * 4096 : kSlot * slots;
    if (need > bytes_) {
        char* fresh = nullptr;
        const hipError_t r = hipHostMalloc((void**)&fresh, need, hipHostMallocCoherent);
        if (r != hipSuccess) return r;
        if (pinned_) (void)hipHostFree(pinned_);
        pinned_ = fresh;
        bytes_ = need;
    }
    for (int k = 0; slots > 1 && k < slots; k++)
        if (!ev_[k]) {
            const hipError_t r = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming);
            if (r != hipSuccess) return r;
        }
    return hipSuccess;
}

// One thread's chunks of a large transfer: k0, k0 + step, ... of the arrays'
// slot-sized pieces, through the slots 2 * k0 and 2 * k0 + 1.
hipError_t StateIo::chunks(bool read, const IoArray* a, int n, size_t k0, size_t step, hipStream_t st) {
    struct Chunk {
        const IoArray* a;
        size_t v0, m;
    };
    size_t next = k0;
    auto take = [&](Chunk& c) {
        size_t k = next;
        for (int i = 0; i < n; i++) {
            const size_t per = kSlot / a[i].bytes(1), have = (a[i].n + per - 1) / per;
            if (k < have) {
                c = {a + i, k * per, std::min(per, a[i].n - k * per)};
                next += step;
                return true;
            }
            k -= have;
        }
        return false;
    };
    char* const slot[2] = {pinned_ + 2 * k0 * kSlot, pinned_ + (2 * k0 + 1) * kSlot};
    hipEvent_t* const ev = ev_ + 2 * k0;
    hipError_t r = hipSuccess;
    Chunk c[2];
    bool have[2] = {false, false};
    auto issue = [&](int s) {
        r = launch(read, c[s].a->comps(), part_of(*c[s].a, c[s].v0, c[s].m), Part{}, slot[s], st);
        if (r == hipSuccess) r = hipEventRecord(ev[s], st);
        have[s] = r == hipSuccess;
    };
    auto host = [&](int s) { return (char*)c[s].a->host + c[s].a->bytes(c[s].v0); };
    if (read && take(c[0])) issue(0);
    for (int s = 0; r == hipSuccess; s ^= 1) {
        if (read) {  // slot s is on its way; start the other, then empty s
            if (!have[s]) break;
            if (take(c[s ^ 1])) issue(s ^ 1);
            if (r != hipSuccess || (r = hipEventSynchronize(ev[s])) != hipSuccess) break;
            memcpy(host(s), slot[s], c[s].a->bytes(c[s].m));
            have[s] = false;
        } else {  // fill s once the device has read it
            if (have[s] && (r = hipEventSynchronize(ev[s])) != hipSuccess) break;
            if (!take(c[s])) break;
            memcpy(slot[s], host(s), c[s].a->bytes(c[s].m));
            issue(s);
        }
    }
    return r;
}

hipError_t StateIo::move(bool read, const IoArray* in, int n, hipStream_t st) {
    const std::lock_guard<std::mutex> hold(lock_);
    IoArray a[2];
    int na = 0;
    bool zeroed = false;
    size_t total = 0;
    for (int i = 0; i < n; i++) {
        if (in[i].n == 0 || !in[i].planes || (read && !in[i].host)) continue;
        if (in[i].host) {
            a[na++] = in[i];
            total += ((size_t)quads_of(in[i].n, in[i].comps())) * 16;
        } else {
            const hipError_t r = hipMemsetAsync(in[i].planes, 0, 3 * sizeof(float) * in[i].n, st);
            if (r != hipSuccess) return r;
            zeroed = true;
        }
    }
    if (na == 0 && !zeroed) return hipSuccess;
    hipError_t r = hipSuccess;
    if (na == 1 && !a[0].w && a[0].bytes(a[0].n) > kCopy && total <= kSlot) {
        if ((r = reserve(total)) != hipSuccess) return r;
        const size_t m = a[0].n, bytes = a[0].bytes(m);
        float *const s = (float*)pinned_, *const h = a[0].host;
        for (size_t i = 0; !read && i < m; i++)
            for (int k = 0; k < 3; k++) s[k * m + i] = h[3 * i + k];
        r = read ? hipMemcpyAsync(s, a[0].planes, bytes, hipMemcpyDeviceToHost, st)
                 : hipMemcpyAsync(a[0].planes, s, bytes, hipMemcpyHostToDevice, st);
        const hipError_t rs = hipStreamSynchronize(st);
        if (r == hipSuccess) r = rs;
        for (size_t i = 0; read && r == hipSuccess && i < m; i++)
            for (int k = 0; k < 3; k++) h[3 * i + k] = s[k * m + i];
        return r;
    }
    if (na > 0 && total <= kSlot) {
        if ((r = reserve(total)) != hipSuccess) return r;
        const Part p0 = part_of(a[0], 0, a[0].n), p1 = na > 1 ? part_of(a[1], 0, a[1].n) : Part{};
        char* const at[2] = {pinned_, pinned_ + 16 * (size_t)p0.quads};
        if (!read)
            for (int i = 0; i < na; i++) memcpy(at[i], a[i].host, a[i].bytes(a[i].n));
        r = launch(read, a[0].comps(), p0, p1, pinned_, st);
        const hipError_t rs = hipStreamSynchronize(st);
        if (r == hipSuccess) r = rs;
        if (read && r == hipSuccess)
            for (int i = 0; i < na; i++) memcpy(a[i].host, at[i], a[i].bytes(a[i].n));
        return r;
    }
    if (na > 0) {
        // (hipStreamPerThread is another stream in every thread: its work is
        // the caller's own thread's)
        const int nt = st == hipStreamPerThread ? 1 : threads_of(total);
        if ((r = reserve(total)) != hipSuccess) return r;
        int dev = 0;
        if ((r = hipGetDevice(&dev)) != hipSuccess) return r;
        hipError_t rt[kThreads] = {};
        std::atomic<int> next(0);
        // shares of the chunks; a thread that cannot be had leaves its share
        // to the others
        auto run = [&]() noexcept {
            for (int k; (k = next.fetch_add(1)) < nt;) rt[k] = chunks(read, a, na, k, nt, st);
        };
        std::thread th[kThreads];
        for (int k = 1; k < nt; k++) try {
                th[k] = std::thread([&]() noexcept {
                    if (hipSetDevice(dev) == hipSuccess) run();
                });
            } catch (...) {
                break;
            }
        run();
        for (std::thread& t : th)
            if (t.joinable()) t.join();
        for (hipError_t e : rt)
            if (r == hipSuccess) r = e;
    }
    // (also after an error: nothing may be on its way to or from the slots)
    const hipError_t rs = hipStreamSynchronize(st);
    return r != hipSuccess ? r : rs;
}

}  // namespace oc
