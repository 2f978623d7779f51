// FP64 direct summation with the reference's softened law, for accuracy
// diagnostics of the tree forces: a_i = sum_j G m_j d / ((r^2 + e0^2) r),
// phi_i = sum_j -(G m_j / e0)(pi/2 - atan(r / e0)), r == 0 pairs skipped
// (Node.cpp:274-276, :301).
//
// Bound by FP64 VALU issue.  One lane takes one target; the sources are
// split over the grid's second dimension so that a few thousand targets still
// fill the chip (16,384 targets alone are 256 waves for 1,024 SIMDs), and
// their coordinates are read through the scalar cache: a source's index is
// the same for the whole wave, so a pair needs no LDS and no barrier.  The
// pair's 1/r and 1/(r^2 + e0^2) come from one reciprocal square root of
// r^2 (r^2 + e0^2)^2, about 21 issue slots with it, and the angle of the
// potential from fp64_math.h, where the correctly rounded square root and
// quotient and the library's atan took ten times that.
//
// The fast pair holds for softening lengths between 2^42 and 2^150 m: there
// no pair's r^2 (r^2 + e0^2)^2 is too small, and one that is too large makes
// its block's sums no numbers, which are formed again with a root and
// quotients of their own.  Other softening lengths test every pair.
//
// A target's sum depends on the sources alone, bit for bit, not on the other
// targets asked for: sources are summed in blocks of fixed length, blocks
// sixteen at a time, those in (at most) four parts of the set, and the parts
// in order, however many of these one wave sums (SumPlan).
//
// 1 M sources, 16,384 targets: with the potential 372 ms one workgroup per 256
// targets, now 26.1; without 212, now 10.5; 300 targets 1.5 and 0.85 ms.
// Against sums in extended precision 2.9e-14 then (a million terms one by one;
// the potential 4.2e-14), now 1.5e-16.
#include <mutex>
#include <type_traits>

#include "ag2_internal.h"
#include "fp64_math.h"

namespace ag2 {
namespace {

constexpr int kDirectBlock = 256;
constexpr int kMid = 16;   // blocks of sources summed at a time

// The order of a target's sum over n sources: blocks of `len` sources, kMid
// blocks at a time, `top` of those at a time, all of them.  A wave sums `per`
// blocks (1, kMid or kMid top): its part of the sum.
struct SumPlan {
    int n, len, blocks, top, per;
};

// Targets: lane k of the grid's first dimension; blocks of sources [split *
// per, ...).  part: column c of split s at (c * splits + s) * nt, unscaled sums.
// ANY: the softening length is outside the fast pair's range.
template <bool POT, bool ANY>
__global__ __launch_bounds__(kDirectBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_direct(SumPlan p, const double *__restrict__ x,
                                                         const double *__restrict__ y, const double *__restrict__ z,
                                                         const double *__restrict__ m, int nt,
                                                         const int64_t *__restrict__ targets,
                                                         const int32_t *__restrict__ inv, double e0,
                                                         double *__restrict__ part) {
    const int k = blockIdx.x * kDirectBlock + threadIdx.x;
    const int split = blockIdx.y;
    const bool valid = k < nt;
    const int64_t i = valid ? inv[targets[k]] : 0;   // caller index -> resident slot
    const double px = x[i], py = y[i], pz = z[i];
    const double e02 = e0 * e0;
    // (all of a target's pairs are long ones, where it is far away itself)
    const bool far = !(fabs(px) < 0x1p150 && fabs(py) < 0x1p150 && fabs(pz) < 0x1p150);
    double gx = 0.0, gy = 0.0, gz = 0.0, ph = 0.0;
    // checked: whatever the pair's scale
    auto pair = [&](int j, auto checked) {
        constexpr bool CHECK = decltype(checked)::value;
        const double dx = x[j] - px, dy = y[j] - py, dz = z[j] - pz;
        // (a pair at r == 0 has d == 0: only its finite factor matters)
        const double r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
        const double s2 = r2 + e02;
        const double mj = r2 != 0.0 ? m[j] : 0.0;
        double f, r = 0.0, ir = 0.0;
        bool ok = true;
        if (!POT) {
            f = m[j] * rsq_full(__builtin_fma(r2 * s2, s2, CHECK ? 0.0 : 1e-290));
            if (CHECK) ok = r2 * s2 * s2 > 0x1p-900 && fabs(f) < 0x1p1000;
        } else {
            ir = rsq_full(fmax(r2, 0x1p-1074));
            r = r2 * ir;
            f = mj * ir * rcp_full(s2);
            if (CHECK) ok = r2 > 0x1p-900 && s2 > 0x1p-900 && s2 < 0x1p300 && fabs(f) < 0x1p1000;
        }
        double ux = dx, uy = dy, uz = dz;
        if (CHECK && __any(!ok)) {
            // the direction first: r^3 alone may leave the range
            const double root = sqrt(r2), inv = r2 != 0.0 ? 1.0 / root : 0.0;
            r = ok ? r : root;
            ir = ok ? ir : inv;
            f = ok ? f : r2 != 0.0 ? mj / s2 : 0.0;
            ux = ok ? dx : dx * inv;
            uy = ok ? dy : dy * inv;
            uz = ok ? dz : dz * inv;
        }
        gx = __builtin_fma(f, ux, gx);
        gy = __builtin_fma(f, uy, gy);
        gz = __builtin_fma(f, uz, gz);
        if (POT) ph = __builtin_fma(mj, softened_angle(e0, r, ir), ph);
    };
    const std::integral_constant<bool, ANY> form;
    double mx = 0.0, my = 0.0, mz = 0.0, mp = 0.0;   // of up to kMid blocks
    double tx = 0.0, ty = 0.0, tz = 0.0, tp = 0.0;   // of those
    const int b1 = (split + 1) * p.per < p.blocks ? (split + 1) * p.per : p.blocks;
    for (int b = split * p.per; b < b1; b++) {
        const int j0 = b * p.len, j1 = p.n - j0 < p.len ? p.n : j0 + p.len;
        gx = gy = gz = ph = 0.0;
        int j = j0;
        for (; j + 4 <= j1; j += 4) { pair(j, form); pair(j + 1, form); pair(j + 2, form); pair(j + 3, form); }
        for (; j < j1; j++) pair(j, form);
        if (!ANY) {
            const bool bad = far || gx != gx || gy != gy || gz != gz || ph != ph;
            if (__any(bad)) {
                const double ox = gx, oy = gy, oz = gz, op = ph;
                gx = gy = gz = ph = 0.0;
                for (int u = j0; u < j1; u++) pair(u, std::true_type{});
                gx = bad ? gx : ox;
                gy = bad ? gy : oy;
                gz = bad ? gz : oz;
                ph = bad ? ph : op;
            }
        }
        mx += gx; my += gy; mz += gz; mp += ph;
        if ((b + 1) % kMid == 0 || b + 1 == b1) {
            tx += mx; ty += my; tz += mz; tp += mp;
            mx = my = mz = mp = 0.0;
        }
    }
    if (!valid) return;
    const size_t col = (size_t)gridDim.y * nt;
    double *out = part + (size_t)split * nt + k;
    out[0] = tx; out[col] = ty; out[2 * col] = tz;
    if (POT) out[3 * col] = tp;
}

// Column c of the result: its parts in the plan's order, scaled.
__global__ __launch_bounds__(256) void k_direct_fold(int nt, int splits, SumPlan p, const double *__restrict__ part,
                                                     double G, double e0, double *ax, double *ay, double *az,
                                                     double *pot) {
    const int k = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
    if (k >= nt) return;
    const double *q = part + (size_t)c * splits * nt + k;
    double s = 0.0, t = 0.0, mid = 0.0;
    for (int u0 = 0; u0 < splits; u0 += kMid) {
        double v[kMid];   // every load before the first sum
#pragma unroll
        for (int k = 0; k < kMid; k++) v[k] = u0 + k < splits ? q[(size_t)(u0 + k) * nt] : 0.0;
#pragma unroll
        for (int k = 0; k < kMid; k++) {
            if (u0 + k >= splits) break;
            const int done = (u0 + k + 1) * p.per;   // blocks so far
            const bool last = u0 + k + 1 == splits;
            mid += v[k];
            if (done % kMid == 0 || last) { t += mid; mid = 0.0; }
            if (done % (kMid * p.top) == 0 || last) { s += t; t = 0.0; }
        }
    }
    double *out = c == 0 ? ax : c == 1 ? ay : c == 2 ? az : pot;
    out[k] = c < 3 ? G * s : -(G / e0) * s;
}

// Blocks of n / 256 sources (a multiple of four, 32 to 256 of them), and at
// most four parts of the whole.
SumPlan sum_plan(int n) {
    SumPlan p;
    p.n = n;
    p.len = ((n + 255) / 256 + 3) / 4 * 4;
    p.len = p.len < 32 ? 32 : p.len > 256 ? 256 : p.len;
    p.blocks = (n + p.len - 1) / p.len;
    p.top = ((p.blocks + kMid - 1) / kMid + 3) / 4;
    p.per = 1;
    return p;
}

// Targets [0, nt) in slices whose parts fit `room` doubles of scratch.  A wave
// takes as many blocks as leave four waves for each of 1,024 SIMDs, or, where
// the scratch holds no more parts, as have to be.
void launch_direct(Ctx &c, int nt, const int64_t *d_targets, int with_pot, double *scratch, size_t room, double *ax,
                   double *ay, double *az, double *pot) {
    const int cols = with_pot ? 4 : 3;
    SumPlan p = sum_plan((int)c.n);
    const int64_t waves = (nt + 63) / 64;
    const int pers[3] = {kMid * p.top, kMid, 1};
    auto parts = [&](int per) { return (int64_t)(p.blocks + per - 1) / per; };
    p.per = pers[0];
    for (int per : pers)
        if (per < p.per && waves * parts(p.per) < 4096 && (int64_t)nt * cols * parts(per) <= (int64_t)room) p.per = per;
    const int splits = (int)parts(p.per);
    const int64_t fit = (int64_t)room / ((int64_t)cols * splits);
    if (fit < 1) throw HipError("no scratch for the direct sum");
    const bool any = !(c.p.e0 >= 0x1p42 && c.p.e0 <= 0x1p150);
    for (int at = 0; at < nt;) {
        const int here = nt - at < fit ? nt - at : (int)fit;
        const dim3 grid(grid_for(here, kDirectBlock), (unsigned)splits), block(kDirectBlock);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, block, 0, c.stream, p, c.x, c.y, c.z, c.m, here, d_targets + at, c.inv,
                               c.p.e0, scratch);
        };
        if (with_pot) any ? go(k_direct<true, true>) : go(k_direct<true, false>);
        else any ? go(k_direct<false, true>) : go(k_direct<false, false>);
        hipLaunchKernelGGL(k_direct_fold, dim3(grid_for(here, 256), cols), dim3(256), 0, c.stream, here, splits, p,
                           scratch, c.p.G, c.p.e0, ax + at, ay + at, az + at, pot ? pot + at : nullptr);
        AG2_HIP(hipGetLastError());
        at += here;
    }
}

}  // namespace

void direct_sum(Ctx &c, int nt, const int64_t *d_targets, double *d_out, int with_pot) {
    build_inverse(c);
    // scratch: the permutation's spare buffers, free between builds
    launch_direct(c, nt, d_targets, with_pot, c.alt[0], (size_t)kStateD * (size_t)c.cap, d_out, d_out + nt,
                  d_out + 2 * (size_t)nt, with_pot ? d_out + 3 * (size_t)nt : nullptr);
}

// ------------------------------------------------ direct sum without allocation
// Scratch of ag2_direct_sum_noalloc: the device copies of the target list
// (int64) and of the four output columns (ax, ay, az, potential), for at most
// AG2_DIRECT_NOALLOC_MAX targets: 5 x 8 B x 65536 = 2.5 MiB per device, held
// until the process ends.  In host code `scratch` is only a stand-in for the
// symbol: its device address, per device, comes from hipGetSymbolAddress.
namespace {
constexpr int64_t kNoAllocTargets = AG2_DIRECT_NOALLOC_MAX;
static __device__ __align__(256) int64_t scratch[kNoAllocTargets * 5];
constexpr int kMaxDevices = 64;
void *g_scratch_addr[kMaxDevices] = {};
std::mutex g_scratch_lock;
}  // namespace

void direct_scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) throw HipError("device ordinal out of range for the direct-sum scratch");
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    if (g_scratch_addr[device]) return;
    // the caller has made `device` current; each device holds its own copy
    void *p = nullptr;
    AG2_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_addr[device] = p;
}

void direct_sum_noalloc(Ctx &c, int nt, const int64_t *h_targets, double *ax, double *ay, double *az, double *pot) {
    void *base = nullptr;
    {
        std::lock_guard<std::mutex> hold(g_scratch_lock);
        base = (c.device >= 0 && c.device < kMaxDevices) ? g_scratch_addr[c.device] : nullptr;
    }
    if (!base) throw HipError("direct-sum scratch of this device was not set up at ag2_create");
    int64_t *d_targets = (int64_t *)base;
    double *d_out = (double *)(d_targets + kNoAllocTargets);
    const size_t bytes = (size_t)nt * 8;
    AG2_HIP(hipMemcpyAsync(d_targets, h_targets, bytes, hipMemcpyHostToDevice, c.stream));
    // the same launches as direct_sum, with the columns kNoAllocTargets apart
    build_inverse(c);
    launch_direct(c, nt, d_targets, pot ? 1 : 0, c.alt[0], (size_t)kStateD * (size_t)c.cap, d_out,
                  d_out + kNoAllocTargets, d_out + 2 * kNoAllocTargets, pot ? d_out + 3 * kNoAllocTargets : nullptr);
    AG2_HIP(hipMemcpyAsync(ax, d_out, bytes, hipMemcpyDeviceToHost, c.stream));
    AG2_HIP(hipMemcpyAsync(ay, d_out + kNoAllocTargets, bytes, hipMemcpyDeviceToHost, c.stream));
    AG2_HIP(hipMemcpyAsync(az, d_out + 2 * kNoAllocTargets, bytes, hipMemcpyDeviceToHost, c.stream));
    if (pot) AG2_HIP(hipMemcpyAsync(pot, d_out + 3 * kNoAllocTargets, bytes, hipMemcpyDeviceToHost, c.stream));
    AG2_HIP(hipStreamSynchronize(c.stream));
}

}  // namespace ag2
