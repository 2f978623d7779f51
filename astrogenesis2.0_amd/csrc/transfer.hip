// Particle state between the caller's host arrays and the device.
//
// The fields of a transfer travel as one flat block: on the device side in
// the permutation's spare buffers (free between builds), packed and unpacked
// by one kernel; on the host side through pinned memory, since a copy to or
// from pageable memory goes through the runtime's own staging on one thread
// (measured here: 7 GB/s into the caller's arrays, against 57 GB/s into
// pinned memory).  A block of up to one piece (4 MiB) is a single copy.  A
// larger one goes piece by piece through a ring of pinned slots (ring.h), and
// a few host threads move the pieces between the ring and the caller's arrays
// while the next ones are under way.  Download of eleven fields of 1 M particles:
// 10-13 ms before, 2.35 ms; the whole state (18 arrays) 9.4-16 ms, 3.5 ms;
// upload of 150,001 particles 1.1 ms.
//
// Pinned buffers are kept for later transfers of any context of the device,
// a few at most, and freed with the device's last context.
#include <functional>
#include <mutex>
#include <vector>

#include "ag2_internal.h"
#include "ring.h"

namespace ag2 {
namespace {

constexpr size_t kPiece = (size_t)4 << 20;
constexpr int kRing = 8;        // pieces of a large transfer's ring
// Host threads beside the caller's.  An upload's first pieces wait for the
// host side, and on a host whose other cores are busy a helper that holds one
// may be off the CPU for milliseconds: below 64 MB the caller alone is as
// fast (20 MB: 1.1 ms) and never waits (3.8 ms with helpers on a busy host).  A
// download of 13 MB takes 0.57 ms with three helpers, 0.82 ms without, one of
// 146 MB 3.5 and 7.8 ms; but on a busy host the small one may wait as well
// (ten steps of 100,000 particles with a download 4.2 ms without helpers, 4.0
// to 7 with), so below 32 MB the caller copies alone there too.
constexpr int kHelpers = 3;
constexpr size_t kHelpDown = (size_t)32 << 20, kHelpUp = (size_t)64 << 20;
constexpr int kMaxDev = 64;
constexpr int kMaxFields = 20;

struct Stage {
    char *host = nullptr;
    int slots = 0;
    hipEvent_t ev[kRing] = {};
};

void stage_free(Stage &s) {
    for (auto &e : s.ev)
        if (e) (void)hipEventDestroy(e);
    if (s.host) (void)hipHostFree(s.host);
    s = Stage{};
}

// Buffers kept for later transfers: up to N of one size.
template <int N>
struct Shelf {
    Stage at[N];
    int n = 0;
    bool take(Stage &s) {
        if (n == 0) return false;
        s = at[--n];
        return true;
    }
    bool give(const Stage &s) {
        if (n == N) return false;
        at[n++] = s;
        return true;
    }
};

struct Kept {
    std::mutex mu;
    int contexts = 0;
    Shelf<4> small;
    Shelf<2> large;
};
Kept &kept(int device) {
    static Kept k[kMaxDev];
    return k[device >= 0 && device < kMaxDev ? device : 0];
}

// The device's pinned buffers for transfers on a stream (Lease, ring.h).
struct Pinned {
    int device;
    bool large;
    hipStream_t stream;
    Stage take() {
        Kept &k = kept(device);
        Stage s;
        {
            std::lock_guard<std::mutex> hold(k.mu);
            if (large ? k.large.take(s) : k.small.take(s)) return s;
        }
        s.slots = large ? kRing : 1;
        try {
            AG2_HIP(hipHostMalloc(&s.host, kPiece * (size_t)s.slots));
            for (int i = 0; i < s.slots; i++) AG2_HIP(hipEventCreateWithFlags(&s.ev[i], hipEventDisableTiming));
        } catch (...) {
            stage_free(s);
            throw;
        }
        return s;
    }
    void drain() { (void)hipStreamSynchronize(stream); }
    bool keep(const Stage &s) {
        Kept &k = kept(device);
        std::lock_guard<std::mutex> hold(k.mu);
        return k.contexts > 0 && (large ? k.large.give(s) : k.small.give(s));
    }
    void destroy(Stage &s) { stage_free(s); }
};

// The device's side of a ring (ring.h): copies on one stream, an event a slot.
struct RingStream {
    Stage &s;
    hipStream_t st;
    std::function<void(int)> copy;   // queue piece p's copy
    void issue(int p) {
        copy(p);
        AG2_HIP(hipEventRecord(s.ev[p % kRing], st));
    }
    void wait(int p) { AG2_HIP(hipEventSynchronize(s.ev[p % kRing])); }
    bool left(int p) {
        const hipError_t e = hipEventQuery(s.ev[p % kRing]);
        if (e == hipErrorNotReady) return false;
        AG2_HIP(e);
        return true;
    }
};

struct PackArgs {
    const double *d[kMaxFields];
    const uint8_t *type;   // after the fields, or null
};

// Resident slot r of field f goes to flat[f n + rid[r]] (caller order).
__global__ __launch_bounds__(256) void k_pack(int n, int nf, int f0, const uint32_t *__restrict__ rid, PackArgs a,
                                              double *__restrict__ flat, uint8_t *__restrict__ tflat) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    const size_t q = rid[r];
    for (int f = 0; f < nf; f++) flat[(size_t)(f0 + f) * n + q] = a.d[f0 + f][r];
    if (tflat) tflat[q] = a.type[r];
}

struct UnpackArgs {
    double *d[kMaxFields];
    int at[kMaxFields];        // column of the flat block, or -1: the default
    double dflt[kMaxFields];
};

// The uploaded columns (and defaults) to the state arrays; every particle
// active, caller order.
__global__ __launch_bounds__(256) void k_unpack(int n, int nf, UnpackArgs a, const double *__restrict__ flat,
                                                const uint8_t *__restrict__ tflat, uint8_t *__restrict__ type,
                                                uint8_t *__restrict__ active, uint32_t *__restrict__ rid) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    for (int f = 0; f < nf; f++) a.d[f][i] = a.at[f] >= 0 ? flat[(size_t)a.at[f] * n + i] : a.dflt[f];
    type[i] = tflat ? tflat[i] : (uint8_t)1;
    active[i] = 1;
    rid[i] = (uint32_t)i;
}

}  // namespace

void transfer_ref(int device) {
    Kept &k = kept(device);
    std::lock_guard<std::mutex> hold(k.mu);
    k.contexts++;
}

void transfer_unref(int device) {
    Kept &k = kept(device);
    Shelf<4> small;
    Shelf<2> large;
    {
        std::lock_guard<std::mutex> hold(k.mu);
        if (--k.contexts > 0) return;
        std::swap(small, k.small);
        std::swap(large, k.large);
    }
    Stage dead;
    while (small.take(dead) || large.take(dead)) stage_free(dead);
}

// Columns src[0 .. nf) (n values each, in resident order) and optionally the
// types, to the caller's arrays in caller order.  Synchronous.
void fields_to_host(Ctx &c, int nf, const double *const *src, double *const *host, const uint8_t *type,
                    uint8_t *htype) {
    const size_t n = (size_t)c.n;
    if (nf > kMaxFields) throw HipError("too many fields in a transfer");
    double *flat = c.alt[0];
    uint8_t *tflat = htype ? (uint8_t *)(flat + (size_t)nf * n) : nullptr;
    std::vector<Run> runs;
    for (int f = 0; f < nf; f++) runs.push_back({(char *)host[f], n * 8});
    if (htype) runs.push_back({(char *)htype, n});
    const size_t bytes = n * 8 * (size_t)nf + (htype ? n : 0);
    if (bytes == 0) return;
    PackArgs a{};
    for (int f = 0; f < nf; f++) a.d[f] = src[f];
    a.type = type;
    const unsigned g = grid_for(c.n, 256);
    auto pack = [&](int f0, int k, bool last) {
        hipLaunchKernelGGL(k_pack, dim3(g), dim3(256), 0, c.stream, (int)n, k, f0, c.rid, a, flat,
                           last ? tflat : nullptr);
        AG2_HIP(hipGetLastError());
    };
    Lease<Stage, Pinned> lease(Pinned{c.device, bytes > kPiece, c.stream});
    Stage &s = lease.buffer;
    if (bytes <= kPiece) {
        pack(0, nf, true);
        AG2_HIP(hipMemcpyAsync(s.host, flat, bytes, hipMemcpyDeviceToHost, c.stream));
        AG2_HIP(hipStreamSynchronize(c.stream));
        lease.whole();
        move_runs(runs, 0, bytes, s.host, true);
        return;
    }
    RingStream dev{s, c.stream, {}};
    Ring<RingStream> ring(dev, s.host, kRing, kPiece, runs, bytes, true, bytes < kHelpDown ? 0 : kHelpers);
    // a few fields at a time, so that the first pieces leave early
    const int per = (int)(n * 8 >= 4 * kPiece ? 1 : 4 * kPiece / (n * 8));
    int packed = 0;
    bool tpacked = !htype;
    dev.copy = [&](int p) {
        const size_t end = ring.off(p) + ring.len(p);
        while ((packed < nf && (size_t)packed * n * 8 < end) || (packed == nf && !tpacked)) {
            const int k = nf - packed < per ? nf - packed : per;
            tpacked = packed + k == nf;
            pack(packed, k, tpacked);
            packed += k;
        }
        AG2_HIP(hipMemcpyAsync(ring.slot(p), (const char *)flat + ring.off(p), ring.len(p), hipMemcpyDeviceToHost,
                               c.stream));
    };
    ring.run();
    AG2_HIP(hipStreamSynchronize(c.stream));
    lease.whole();
}

// The caller's columns to the state arrays: dst[f] from host[f], or filled
// with dflt[f] where host[f] is null; types (1 where htype is null), every
// particle active, resident order = caller order.  Synchronous.
void fields_to_device(Ctx &c, int nf, double *const *dst, const double *const *host, const double *dflt,
                      const uint8_t *htype) {
    const size_t n = (size_t)c.n;
    if (nf > kMaxFields) throw HipError("too many fields in a transfer");
    double *flat = c.alt[0];
    UnpackArgs a{};
    std::vector<Run> runs;
    int cols = 0;
    for (int f = 0; f < nf; f++) {
        a.d[f] = dst[f];
        a.at[f] = host[f] ? cols : -1;
        a.dflt[f] = dflt[f];
        if (host[f]) {
            runs.push_back({(char *)const_cast<double *>(host[f]), n * 8});
            cols++;
        }
    }
    if (cols >= kStateD) throw HipError("too many columns in a transfer");   // the types follow the columns
    uint8_t *tflat = htype ? (uint8_t *)(flat + (size_t)cols * n) : nullptr;
    if (htype) runs.push_back({(char *)const_cast<uint8_t *>(htype), n});
    const size_t bytes = n * 8 * (size_t)cols + (htype ? n : 0);
    auto unpack = [&]() {
        hipLaunchKernelGGL(k_unpack, dim3(grid_for(c.n, 256)), dim3(256), 0, c.stream, (int)n, nf, a, flat, tflat,
                           c.type, c.active, c.rid);
        AG2_HIP(hipGetLastError());
    };
    if (bytes == 0) return unpack();
    Lease<Stage, Pinned> lease(Pinned{c.device, bytes > kPiece, c.stream});
    Stage &s = lease.buffer;
    if (bytes <= kPiece) {
        move_runs(runs, 0, bytes, s.host, false);
        AG2_HIP(hipMemcpyAsync(flat, s.host, bytes, hipMemcpyHostToDevice, c.stream));
    } else {
        RingStream dev{s, c.stream, {}};
        Ring<RingStream> ring(dev, s.host, kRing, kPiece, runs, bytes, false, bytes < kHelpUp ? 0 : kHelpers);
        dev.copy = [&](int p) {
            AG2_HIP(hipMemcpyAsync((char *)flat + ring.off(p), ring.slot(p), ring.len(p), hipMemcpyHostToDevice,
                                   c.stream));
        };
        ring.run();
    }
    unpack();
    AG2_HIP(hipStreamSynchronize(c.stream));
    lease.whole();
}

}  // namespace ag2
