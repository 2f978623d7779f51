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
// targets asked for: sources are summed in blocks of fixed length, and the
// blocks in a binary tree (pairs of neighbours, pairs of those, a node without
// a right half being its left one), of which a workgroup takes a node of any
// level, as the number of targets and the scratch for the nodes' sums leave it.
// Its four waves take a quarter of the node each, for the same 64 targets.
// 1 M sources, 16,384 targets: 372 ms with the potential and 212 without by one
// workgroup per 256 targets, now 26.1 and 10.5; 256 targets 0.71 and 0.30 ms.
// (A node per wave, four times the parts: 40,000 sources, 16,384 targets, whose
// parts the scratch bounds, 1.69 ms, now 1.35.)
// Against sums in extended precision 2.9e-14 then (a million terms one by one;
// the potential 4.2e-14), now 1.1e-16.
#include <mutex>
#include <type_traits>

#include "ag2_internal.h"
#include "fp64_math.h"

namespace ag2 {
namespace {

constexpr int kDirectWaves = 4;
constexpr int kLevels = 24;   // of the tree over blocks

// Sources in blocks of `len`; a workgroup sums 2^level (level >= 2) of them.
struct SumPlan {
    int n, len, blocks, level;
};

// Targets: 64 per workgroup of the grid's first dimension, a lane each; blocks of
// sources from split 2^level on, a quarter of them per wave.  part: column c of
// split s at (c * splits + s) * nt, unscaled sums.
// ANY: the softening length is outside the fast pair's range.
template <bool POT, bool ANY>
__global__ __launch_bounds__(64 * kDirectWaves) __attribute__((amdgpu_waves_per_eu(4))) void
k_direct(SumPlan p, const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
         const double *__restrict__ m, int nt, const int64_t *__restrict__ targets, const int32_t *__restrict__ inv,
         double e0, double *__restrict__ part) {
    __shared__ double quarter[kDirectWaves][4][64];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int k = blockIdx.x * 64 + lane;
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
        if (POT) ph = __builtin_fma(mj, softened_angle_own(e0, r, ir), ph);
    };
    const std::integral_constant<bool, ANY> form;
    double node[kLevels][4];   // left halves that wait for their right ones, by level
    const int size = 1 << (p.level - 2);   // blocks of a quarter
    const int b0 = (split << p.level) + wave * size, b1 = b0 + size < p.blocks ? b0 + size : p.blocks;
    for (int b = b0; b < b1; b++) {
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
        int l = 0;
        for (; (b - b0) >> l & 1; l++) {
            gx = node[l][0] + gx;
            gy = node[l][1] + gy;
            gz = node[l][2] + gz;
            if (POT) ph = node[l][3] + ph;
        }
        node[l][0] = gx; node[l][1] = gy; node[l][2] = gz;
        if (POT) node[l][3] = ph;
    }
    if (b0 < b1) {
        // what is left of an incomplete node, the set's last
        const int done = b1 - b0;
        int l = __builtin_ctz(done);
        gx = node[l][0]; gy = node[l][1]; gz = node[l][2];
        if (POT) ph = node[l][3];
        for (l++; done >> l; l++)
            if (done >> l & 1) {
                gx = node[l][0] + gx;
                gy = node[l][1] + gy;
                gz = node[l][2] + gz;
                if (POT) ph = node[l][3] + ph;
            }
    }
    quarter[wave][0][lane] = gx;
    quarter[wave][1][lane] = gy;
    quarter[wave][2][lane] = gz;
    if (POT) quarter[wave][3][lane] = ph;
    __syncthreads();
    // wave c: column c of the quarters that there are
    if (!valid || wave >= (POT ? 4 : 3)) return;
    const int rest = p.blocks - (split << p.level);
    const double lo = quarter[0][wave][lane], hi = quarter[2][wave][lane];
    double sum = rest > size ? lo + quarter[1][wave][lane] : lo;
    if (rest > 2 * size) sum = sum + (rest > 3 * size ? hi + quarter[3][wave][lane] : hi);
    part[((size_t)wave * gridDim.y + split) * nt + k] = sum;
}

// Column c of the result: its parts up the rest of the tree, scaled.
__global__ __launch_bounds__(256) void k_direct_fold(int nt, int splits, const double *__restrict__ part, double G,
                                                     double e0, double *ax, double *ay, double *az, double *pot) {
    constexpr int kAt = 16;   // parts read at a time
    const int k = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
    if (k >= nt) return;
    const double *q = part + (size_t)c * splits * nt + k;
    double node[kLevels];
    const int all = (splits + kAt - 1) / kAt;
    double s = 0.0;
    for (int b = 0; b < all; b++) {
        const int have = splits - b * kAt;
        double v[kAt];
#pragma unroll
        for (int u = 0; u < kAt; u++) v[u] = u < have ? q[(size_t)(b * kAt + u) * nt] : 0.0;
#pragma unroll
        for (int d = 1; d < kAt; d *= 2)
#pragma unroll
            for (int u = 0; u < kAt; u += 2 * d) v[u] = u + d < have ? v[u] + v[u + d] : v[u];
        s = v[0];
        int l = 0;
        for (; b >> l & 1; l++) s = node[l] + s;
        node[l] = s;
    }
    int l = __builtin_ctz(all);
    s = node[l];
    for (l++; all >> l; l++)
        if (all >> l & 1) s = node[l] + s;
    double *out = c == 0 ? ax : c == 1 ? ay : c == 2 ? az : pot;
    out[k] = c < 3 ? G * s : -(G / e0) * s;
}

// Targets [0, nt) in slices whose parts fit `room` doubles of scratch.  Blocks
// of n / 256 sources (a multiple of four, 32 to 256 of them).  Parts: up to 64
// waves for each of 1,024 SIMDs (with 16, four rounds of them, 16,384 targets
// waited 30.3 ms for the last, with 64 27.7), of at least 1,024 sources.
void launch_direct(Ctx &c, int nt, const int64_t *d_targets, int with_pot, double *scratch, size_t room, double *ax,
                   double *ay, double *az, double *pot) {
    const int cols = with_pot ? 4 : 3;
    SumPlan p;
    p.n = (int)c.n;
    p.len = ((p.n + 255) / 256 + 3) / 4 * 4;
    p.len = p.len < 32 ? 32 : p.len > 256 ? 256 : p.len;
    p.blocks = (p.n + p.len - 1) / p.len;
    const bool any = !(c.p.e0 >= 0x1p42 && c.p.e0 <= 0x1p150);
    for (int at = 0; at < nt;) {
        const size_t fit = room / (size_t)cols;
        const int here = (size_t)(nt - at) < fit ? nt - at : (int)fit;
        if (here < 1) throw HipError("no scratch for the direct sum");
        const int64_t waves = (here + 63) / 64 * kDirectWaves;
        int64_t most = (65536 + waves - 1) / waves;
        if (most > (p.n + 1023) / 1024) most = (p.n + 1023) / 1024;
        if (most > (int64_t)(fit / (size_t)here)) most = (int64_t)(fit / (size_t)here);
        if (most > 65535) most = 65535;
        p.level = 2;
        while (((p.blocks - 1) >> p.level) + 1 > most) p.level++;
        const int splits = ((p.blocks - 1) >> p.level) + 1;
        const dim3 grid(grid_for(here, 64), (unsigned)splits), block(64 * kDirectWaves);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, block, 0, c.stream, p, c.x, c.y, c.z, c.m, here, d_targets + at, c.inv,
                               c.p.e0, scratch);
        };
        if (with_pot) any ? go(k_direct<true, true>) : go(k_direct<true, false>);
        else any ? go(k_direct<false, true>) : go(k_direct<false, false>);
        hipLaunchKernelGGL(k_direct_fold, dim3(grid_for(here, 256), cols), dim3(256), 0, c.stream, here, splits,
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
