// Octree build on the device: root half-width, octant keys, a key sort chosen
// by size (merge, sample or LSD radix), tie refinement, linear-octree topology
// from the levels that neighbouring keys share, node sums over each node's own
// particle range.  Replaces Tree::buildTree / Node::insert (Tree.cpp:24-55,
// Node.cpp:405-699).  Integer and FP64 streaming work: bound by HBM in the
// millions, by launches and chains of dependent reads below.
#include "ag2_internal.h"

namespace ag2 {
namespace {

constexpr unsigned long long kOut = ~0ull;

// ------------------------------------------------------------ tree width
// (k_kick_drift forms the same partials in a step of up to 256 kTwBlocks
// particles.)
__global__ __launch_bounds__(256) void k_tw_partial(int n, const double *__restrict__ x,
                                                    const double *__restrict__ y,
                                                    const double *__restrict__ z, double *part) {
    double s = 0.0, q = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        double d = sqrt(x[i] * x[i] + y[i] * y[i] + z[i] * z[i]);
        s += d;
        q += d * d;
    }
    tw_block_sums(s, q, part);
}

// Tree::calcTreeWidth (Tree.cpp:86-117): cut = mean + 10 sigma of |x|,
// then the largest |x| within the cut.  Every workgroup folds the sum
// partials itself in the same fixed order (so all get the same cut, and
// workgroup 0 records it), then writes the maximum of its particles.
__global__ __launch_bounds__(256) void k_tw_max(int n, const double *__restrict__ x, const double *__restrict__ y,
                                                const double *__restrict__ z, int nb, const double *tw,
                                                DevState *ds, unsigned long long *part) {
    __shared__ unsigned long long wmax[4];
    __shared__ double ls[4], lq[4], scut;
    {
        double s = 0.0, q = 0.0;
        for (int b = threadIdx.x; b < nb; b += 256) { s += tw[2 * b]; q += tw[2 * b + 1]; }
        s = wave_sum(s);
        q = wave_sum(q);
        int w = threadIdx.x >> 6;
        if (lane_id() == 0) { ls[w] = s; lq[w] = q; }
        __syncthreads();
        if (threadIdx.x == 0) {
            double sum = ((ls[0] + ls[1]) + ls[2]) + ls[3];
            double sq = ((lq[0] + lq[1]) + lq[2]) + lq[3];
            double mean = sum / (double)n;
            double sd = sqrt(sq / (double)n - mean * mean);
            scut = mean + 10.0 * sd;
            if (blockIdx.x == 0) {
                ds->sum = sum;
                ds->sumsq = sq;
                ds->cut = scut;
                ds->gap = 0ull;
                ds->err = 0;
                ds->max_level = 0;
                ds->tie_big = 0;
                ds->tie_deep = 0;
                ds->any_bucket = 0;
                ds->max_prefix_run = 0;
            }
        }
        __syncthreads();
    }
    double cut = scut;
    unsigned long long best = 0ull;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        double d = sqrt(x[i] * x[i] + y[i] * y[i] + z[i] * z[i]);
        if (d <= cut) {
            unsigned long long b = (unsigned long long)__double_as_longlong(d);
            best = b > best ? b : best;
        }
    }
    for (int o = 32; o >= 1; o >>= 1) {
        unsigned long long t = __shfl_xor(best, o, 64);
        best = t > best ? t : best;
    }
    if (lane_id() == 0) wmax[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = wmax[0];
        for (int w = 1; w < 4; w++) b = wmax[w] > b ? wmax[w] : b;
        part[blockIdx.x] = b;
    }
}

// ------------------------------------------------------------ keys
// Every workgroup first folds the per-workgroup maxima of k_tw_max into R
// (workgroup 0 records it).  All but a few particles in a million stand clear
// of every cell face and take their key from the scaled position; the
// reference's descent through 21 levels of centres and bounds, run for every
// particle, made this 27 us at 1,000,000 particles (now 11) and 94 us at
// 4,000,000 (32).
__global__ __launch_bounds__(256) void k_keygen(int n, const double *__restrict__ x, const double *__restrict__ y,
                                                const double *__restrict__ z, int nb,
                                                const unsigned long long *rmax, DevState *ds,
                                                uint64_t *key, uint32_t *idx, uint8_t *gapl) {
    __shared__ unsigned long long w4[4];
    // the position is loaded first: its loads are in flight while R is folded
    const int i = blockIdx.x * 256 + threadIdx.x;
    double px = 0.0, py = 0.0, pz = 0.0;
    if (i < n) { px = x[i]; py = y[i]; pz = z[i]; }
    unsigned long long v = 0ull;
    for (int k = threadIdx.x; k < nb; k += 256) v = rmax[k] > v ? rmax[k] : v;
    for (int o = 32; o >= 1; o >>= 1) {
        unsigned long long q = __shfl_xor(v, o, 64);
        v = q > v ? q : v;
    }
    if (lane_id() == 0) w4[threadIdx.x >> 6] = v;
    __syncthreads();
    unsigned long long rb = w4[0];
    for (int w = 1; w < 4; w++) rb = w4[w] > rb ? w4[w] : rb;
    if (blockIdx.x == 0 && threadIdx.x == 0) ds->Rbits = rb;
    if (i >= n) return;
    double R = __longlong_as_double((long long)rb);
    uint64_t k1 = 0ull, k2;
    int g = 0;
    bool in = !(px < -R || px > R || py < -R || py > R || pz < -R || pz > R);
    if (in && !core::octant_word0_apart(px, py, pz, 1048576.0 / R, &k1))
        in = core::octant_path(px, py, pz, R, 21, &k1, &k2, &g);
    key[i] = in ? k1 : kOut;
    idx[i] = (uint32_t)i;
    gapl[i] = in ? (uint8_t)g : (uint8_t)255;
}

// ------------------------------------------------------------ radix sort
// Workgroup tile: kSortTile keys, kSortItems per thread; wave w owns tile
// positions [64 kSortItems w, 64 kSortItems (w + 1)), item j of lane l at
// 64 kSortItems w + 64 j + l, so (wave, item, lane) is tile order and the
// scatter is stable.
constexpr int kSortItems = kSortTile / 256;
constexpr int kSortSmallTiles = 16;   // up to this many tiles the scatter forms its own offsets
__device__ __forceinline__ void rs_hist_tile(int n, const uint64_t *__restrict__ key, int shift, uint32_t *hist,
                                             int nblk, int tile) {
    __shared__ uint32_t cnt[256];
    int w = threadIdx.x >> 6;
    int base = tile * kSortTile + w * (64 * kSortItems) + lane_id();
    // the keys are loaded before the counters are cleared: the loads are in
    // flight across the barrier
    int dg[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        int pos = base + j * 64;
        dg[j] = pos < n ? (int)((key[pos] >> shift) & 255) : -1;
    }
    cnt[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; j++)
        if (dg[j] >= 0) atomicAdd(&cnt[dg[j]], 1u);
    __syncthreads();
    hist[threadIdx.x * nblk + tile] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(256) void k_rs_hist(int n, const uint64_t *__restrict__ key, int shift,
                                                 uint32_t *hist, int nblk) {
    rs_hist_tile(n, key, shift, hist, nblk, blockIdx.x);
}

// One workgroup per digit: exclusive scan of that digit's per-tile counts.
__device__ __forceinline__ void rs_scan_digit(int nblk, uint32_t *hist, uint32_t *dtotal, int digit) {
    __shared__ int scr[4];
    uint32_t *h = hist + (size_t)digit * nblk;
    int per = (nblk + 255) / 256;
    int s0 = threadIdx.x * per;
    int s1 = s0 + per < nblk ? s0 + per : nblk;
    int local = 0;
    for (int k = s0; k < s1; k++) local += (int)h[k];
    int tot;
    int run = block256_excl_scan(local, scr, &tot);
    for (int k = s0; k < s1; k++) {
        int t = (int)h[k];
        h[k] = (uint32_t)run;
        run += t;
    }
    if (threadIdx.x == 0) dtotal[digit] = (uint32_t)tot;
}

__global__ __launch_bounds__(256) void k_rs_scan(int nblk, uint32_t *hist, uint32_t *dtotal) {
    rs_scan_digit(nblk, hist, dtotal, blockIdx.x);
}

// SMALL: hist holds the raw per-tile counts (no k_rs_scan pass) and each
// workgroup forms its own offsets from them -- nblk reads per digit, cheap
// for the few tiles of a small particle set, and one launch fewer per pass.
template <bool SMALL>
__device__ __forceinline__ void rs_scatter_tile(int n, const uint64_t *__restrict__ kin,
                                                const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
                                                uint32_t *__restrict__ vout, int shift,
                                                const uint32_t *__restrict__ hist,
                                                const uint32_t *__restrict__ dtotal, int nblk, int tile) {
    __shared__ int sbase[256];
    __shared__ int wcnt[4][256];
    __shared__ int scr[4];
    int tid = threadIdx.x;
    int tot;
    int w = tid >> 6;
    int base = tile * kSortTile + w * (64 * kSortItems) + lane_id();
    // the tile's keys are loaded first: the offsets below do not need them,
    // so the loads are in flight while the offsets are formed
    uint64_t keys[kSortItems];
    uint32_t vals[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        const int pos = base + j * 64;
        keys[j] = pos < n ? kin[pos] : 0ull;
        vals[j] = pos < n ? vin[pos] : 0u;
    }
    if (SMALL) {
        const uint32_t *h = hist + (size_t)tid * nblk;
        int before = 0, all = 0;
        for (int t = 0; t < nblk; t++) {
            const int v = (int)h[t];
            before += t < tile ? v : 0;
            all += v;
        }
        int ex = block256_excl_scan(all, scr, &tot);
        sbase[tid] = ex + before;
    } else {
        int ex = block256_excl_scan((int)dtotal[tid], scr, &tot);
        sbase[tid] = ex + (int)hist[tid * nblk + tile];
    }
    wcnt[0][tid] = 0; wcnt[1][tid] = 0; wcnt[2][tid] = 0; wcnt[3][tid] = 0;
    __syncthreads();
    unsigned long long below = lanes_below();
    int loc[kSortItems], dig[kSortItems];
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        int pos = base + j * 64;
        bool valid = pos < n;
        const uint64_t k = keys[j];
        int d = (int)((k >> shift) & 255);
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            int bit = (d >> b) & 1;
            unsigned long long bm = __ballot(bit);
            peers &= bit ? bm : ~bm;
        }
        if (!valid) peers = 0ull;
        int rank = __popcll(peers & below);
        int cur = valid ? wcnt[w][d] : 0;
        if (valid && (peers & below) == 0ull) wcnt[w][d] = cur + __popcll(peers);
        loc[j] = valid ? cur + rank : -1; dig[j] = d;
    }
    __syncthreads();
    {
        int s = 0;
        for (int k = 0; k < 4; k++) { int t = wcnt[k][tid]; wcnt[k][tid] = s; s += t; }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortItems; j++) {
        if (loc[j] >= 0) {
            int dst = sbase[dig[j]] + wcnt[w][dig[j]] + loc[j];
            kout[dst] = keys[j];
            vout[dst] = vals[j];
        }
    }
}

template <bool SMALL>
__global__ __launch_bounds__(256) void k_rs_scatter(int n, const uint64_t *__restrict__ kin,
                                                    const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
                                                    uint32_t *__restrict__ vout, int shift,
                                                    const uint32_t *__restrict__ hist,
                                                    const uint32_t *__restrict__ dtotal, int nblk) {
    rs_scatter_tile<SMALL>(n, kin, vin, kout, vout, shift, hist, dtotal, nblk, blockIdx.x);
}

// ------------------------------------------------------------ merge sort
// Two launches for a set of a few tiles, where the radix passes are launches
// and little else (six bytes are 18 launches of 4-7 us).  k_ms_tile
// sorts each tile of TILE keys by itself in LDS (stable radix passes over
// the bytes the build sorts, bound by their barriers and LDS round trips:
// 2.5 us each); k_ms_merge gives each key its place: its
// position in its own tile plus, for every other tile, the number of keys
// that come before it, by binary search (equal keys in tile order, so the
// sort is stable).  A tile whose range leaves out a whole wave's keys is not
// searched: particles move little between steps, so most are.
constexpr int kMsThreads = 1024;
constexpr int kMsWaves = kMsThreads / 64;
// Sort phase in microseconds (first build after an upload, in caller order;
// later builds are 1-5 us below), radix passes / merge with tiles of 2048 /
// of 4096 / sample sort (merge with tiles of 1024: 10,000 26, 15,000 27 for
// 36, 20,000 40 for 37 -- past the 16 tiles a key's four lanes take in one
// round):
//    10,000   69 / 33 / 36 / 51        100,003   89 / 142 / 95 / 56
//    20,000   73 / 36 / 43 / 51        200,000   94 / 467 / 273 / 69
//    33,333   86 / 42 / 46 / 52        520,000  112 / - / - / 84
//    45,000   87 / 52 / 48 / 52      1,000,000  146 / - / - / 108
//    65,000   87 / 66 / 55 / 53      1,500,000  181 / - / - / 182
//                                    2,000,000  217 / - / - / 211
//                                    3,000,000  288 / - / - / 366
// The merge's searches grow with the tiles' number for every key; the sample
// sort fills a CU with each workgroup, and past two rounds of 256 tiles the
// ranks of the samples cost too (later builds: 1,500,000 178 against 167,
// 2,000,000 216 against 190, 3,000,000 287 against 317).
constexpr int kMsTiny = 16384, kMsSmall = 40000, kMsMax = 60000;   // merge: up to here kMsTiny0, kMsTile0, kMsTile1
constexpr int kMsTiny0 = 1024;
constexpr int kMsTile0 = 2048, kMsTile1 = 4096;
constexpr int kBsTiles = 512;                         // most tiles of a set (a thread each)
constexpr int kBsMax = kBsTiles * kMsTile1;           // sample sort up to here, radix passes above
constexpr int kBsBatchMax = kBsTiles * kMsTile0;      // ... in a batch, whose tiles are the smaller ones

// The first sample of a tile: its number's bits reversed, within the step.
__device__ inline int sample_phase(int tile, int step) {
    return (int)(__brev((unsigned)tile) >> (__builtin_clz((unsigned)step) + 1)) & (step - 1);
}

// Stable sort of len keys by one workgroup in LDS, on the bytes lo .. 7 in
// which they differ at all.  Item j of lane l of wave w holds position
// (w it + j) 64 + l before and after (it: items in use, 1024 it >= len).
template <int ITEMS>
struct SortLds {
    uint64_t k[ITEMS * kMsThreads];
    uint32_t v[ITEMS * kMsThreads];
    int wcnt[kMsWaves][256];
    int wtot[4];
    unsigned long long red[kMsWaves];
};

template <int ITEMS>
__device__ __forceinline__ void lds_sort(SortLds<ITEMS> &S, uint64_t (&k)[ITEMS], uint32_t (&v)[ITEMS], int it,
                                         int len, int lo) {
    const int tid = threadIdx.x, w = tid >> 6, lane = lane_id();
    const int base = w * (64 * it) + lane;
    // the bits in which the keys differ; unused positions get a key with all
    // of them set, which stays behind (the sort is stable)
    if (tid == 0) S.red[0] = k[0];
    __syncthreads();
    const unsigned long long k0 = S.red[0];
    unsigned long long diff = 0ull;
#pragma unroll
    for (int j = 0; j < ITEMS; j++)
        if (j < it && base + j * 64 < len) diff |= k[j] ^ k0;
    for (int d = 32; d >= 1; d >>= 1) diff |= __shfl_xor(diff, d, 64);
    __syncthreads();
    if (lane == 0) S.red[w] = diff;
    __syncthreads();
    diff = 0ull;
    for (int u = 0; u < kMsWaves; u++) diff |= S.red[u];
#pragma unroll
    for (int j = 0; j < ITEMS; j++)
        if (j < it && base + j * 64 >= len) { k[j] = k0 | diff; v[j] = 0u; }
    const unsigned long long below = lanes_below();
    for (int pass = lo; pass < 8; pass++) {
        if ((diff >> (8 * pass) & 255) == 0) continue;
        for (int d = lane; d < 256; d += 64) S.wcnt[w][d] = 0;
        wave_sync_lds();
        int loc[ITEMS], dig[ITEMS];
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (j >= it) break;
            const int d = (int)((k[j] >> (8 * pass)) & 255);
            unsigned long long peers = ~0ull;
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const int bit = (d >> b) & 1;
                const unsigned long long bm = __ballot(bit);
                peers &= bit ? bm : ~bm;
            }
            const int cur = S.wcnt[w][d];
            wave_sync_lds();
            if ((peers & below) == 0ull) S.wcnt[w][d] = cur + __popcll(peers);
            wave_sync_lds();
            loc[j] = cur + __popcll(peers & below);
            dig[j] = d;
        }
        __syncthreads();
        // digit d's first place: the keys of smaller digits, then of earlier waves
        int inc = 0, tot = 0;
        if (tid < 256) {
            for (int u = 0; u < kMsWaves; u++) tot += S.wcnt[u][tid];
            inc = wave_incl_scan(tot);
            if (lane == 63) S.wtot[w] = inc;
        }
        __syncthreads();
        if (tid < 256) {
            int at = inc - tot;
            for (int u = 0; u < w; u++) at += S.wtot[u];
            for (int u = 0; u < kMsWaves; u++) { const int c = S.wcnt[u][tid]; S.wcnt[u][tid] = at; at += c; }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (j >= it) break;
            const int to = S.wcnt[w][dig[j]] + loc[j];
            S.k[to] = k[j];
            S.v[to] = v[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            if (j >= it) break;
            k[j] = S.k[base + j * 64];
            v[j] = S.v[base + j * 64];
        }
        // (the next pass writes S.k only after two more barriers)
    }
}

template <int TILE>
__device__ __forceinline__ void ms_tile(int n, const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                        uint64_t *__restrict__ kout, uint32_t *__restrict__ vout, int lo, int tile,
                                        uint64_t *__restrict__ samp, int step) {
    constexpr int kMsItems = TILE / kMsThreads;
    __shared__ SortLds<kMsItems> S;
    const int t0 = tile * TILE;
    const int len = n - t0 < TILE ? n - t0 : TILE;
    const int base = (threadIdx.x >> 6) * (64 * kMsItems) + lane_id();
    uint64_t k[kMsItems];
    uint32_t v[kMsItems];
#pragma unroll
    for (int j = 0; j < kMsItems; j++) {
        const int p = base + j * 64;
        k[j] = p < len ? kin[t0 + p] : 0ull;
        v[j] = p < len ? vin[t0 + p] : 0u;
    }
    lds_sort<kMsItems>(S, k, v, kMsItems, len, lo);
    const int phase = step ? sample_phase(tile, step) : 0;
#pragma unroll
    for (int j = 0; j < kMsItems; j++) {
        const int p = base + j * 64;
        if (p < len) {
            kout[t0 + p] = k[j];
            vout[t0 + p] = v[j];
            if (step && (p & (step - 1)) == phase) samp[tile * (TILE / step) + p / step] = k[j] >> (8 * lo);
        }
    }
}

// Element i of the tile-sorted keys to its place: kMsLanes neighbouring lanes
// per element share the other tiles, four at a time each, searched side by
// side (one lane for all of them waits out every search in turn).
constexpr int kMsLanes = 4;
constexpr int kMsPer = 256 / kMsLanes;   // elements per workgroup

template <int TILE>
__device__ __forceinline__ void ms_merge(int n, const uint64_t *__restrict__ kin, const uint32_t *__restrict__ vin,
                                         uint64_t *__restrict__ kout, uint32_t *__restrict__ vout, int lo, int i) {
    constexpr int kG = 4;
    const bool on = i < n;
    const int e = on ? i : n - 1;
    const int shift = 8 * lo;
    const uint64_t k = kin[e], q = k >> shift;
    const int own = e / TILE, tiles = (n + TILE - 1) / TILE;
    const int share = threadIdx.x & (kMsLanes - 1);
    int at = share == 0 ? e - own * TILE : 0;
    for (int t0 = 0; t0 < tiles; t0 += kG * kMsLanes) {
        const int t = t0 + share * kG;
        int len[kG], pos[kG];
        bool need = false;
#pragma unroll
        for (int u = 0; u < kG; u++) {
            const int b = (t + u) * TILE;
            len[u] = t + u < tiles && t + u != own ? (n - b < TILE ? n - b : TILE) : 0;
            pos[u] = 0;
            if (len[u] > 0) {
                const uint64_t first = kin[b] >> shift, last = kin[b + len[u] - 1] >> shift;
                const bool before = t + u < own;   // equal keys there come first
                const bool all = before ? last <= q : last < q, none = before ? first > q : first >= q;
                pos[u] = all ? len[u] : 0;
                need |= !all && !none;
            }
        }
        if (__any(need)) {
#pragma unroll
            for (int u = 0; u < kG; u++) pos[u] = 0;
            for (int step = TILE; step; step >>= 1)
#pragma unroll
                for (int u = 0; u < kG; u++) {
                    const int p = pos[u] + step;
                    if (p <= len[u]) {
                        const uint64_t o = kin[(t + u) * TILE + p - 1] >> shift;
                        if (t + u < own ? o <= q : o < q) pos[u] = p;
                    }
                }
        }
#pragma unroll
        for (int u = 0; u < kG; u++) at += pos[u];
    }
    for (int d = kMsLanes / 2; d >= 1; d >>= 1) at += __shfl_xor(at, d, 64);
    if (on && share == 0) { kout[at] = k; vout[at] = vin[e]; }
}

// ------------------------------------------------------------ sample sort
// Three launches for a set between the merge sort's range and that of the
// radix passes (18 launches, bandwidth only in the millions): k_ms_tile leaves every step-th key of its sorted tile as a
// sample; k_bs_split ranks the samples among all of them and keeps every 64th
// as a splitter;
// k_bs_bucket finds one bucket's piece of every tile, gathers the pieces in
// tile order and sorts them in LDS.  Splitters are single elements (key,
// tile, position), so equal keys part in the stable order and long runs of
// them split like any others.
// The samples of tile t stand at t's own phase of the step (its number with
// the bits reversed): samples at the same quantiles of tiles that hold like
// mixtures of keys (any order but a sorted one) would fall in clusters, with
// hardly a splitter between them.  A bucket holds 64 steps on average and
// strays by an eighth of that (one standard deviation, for a random order);
// the room is twice the average, and k_bs_bucket ranks the keys of a larger
// one singly.
constexpr int kBsPer = 64;   // samples per bucket

struct Splitter {
    uint64_t q;       // key from the lowest sorted bit on
    int tile, pos;
};

__device__ inline int sample_count(int n, int TILE, int tile, int step) {
    const int len = n - tile * TILE < TILE ? n - tile * TILE : TILE;
    const int ph = sample_phase(tile, step);
    return len > ph ? ((len - ph - 1) >> (__builtin_ctz((unsigned)step))) + 1 : 0;
}

// Elements of tile u that come before q of tile t (t != u): its sorted keys
// below q, and those equal to q if u comes first.
__device__ inline bool before(uint64_t o, uint64_t q, bool first) { return first ? o <= q : o < q; }

// The samples of one tile, a lane each: their ranks, and the splitters among
// them.  The workgroup's waves share the other tiles, whose samples they
// search in LDS, four lists side by side (7 us at 100,000 disk particles, 14
// at 1,000,000, once lists that lie wholly to one side are left out; 12 and
// 22 with every list searched, up to 99 where each sample searched the lists
// in memory).
template <int TILE>
__device__ __forceinline__ void bs_split(int n, int step, const uint64_t *__restrict__ samp, Splitter *split,
                                         int own) {
    constexpr int kG = 4;
    __shared__ uint64_t list[kG * kMsThreads];
    __shared__ int part[kMsThreads];
    const int S = TILE / step, groups = S / 64;       // waves that hold the tile's samples
    const int tiles = (n + TILE - 1) / TILE;
    const int w = threadIdx.x >> 6, mine = w % groups, slot = w / groups, slots = kMsWaves / groups;
    const int j = mine * 64 + lane_id();
    const bool on = j < sample_count(n, TILE, own, step);
    const uint64_t q = on ? samp[(size_t)own * S + j] : 0ull;
    int at = 0;
    for (int t0 = 0; t0 < tiles; t0 += slots * kG) {
        const int t = t0 + slot * kG;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kG; u++)
            if (t + u < tiles) list[(slot * kG + u) * S + j] = samp[(size_t)(t + u) * S + j];
        __syncthreads();
        int len[kG], pos[kG];
        bool need = false;
#pragma unroll
        for (int u = 0; u < kG; u++) {
            len[u] = t + u < tiles && t + u != own ? sample_count(n, TILE, t + u, step) : 0;
            pos[u] = 0;
            if (len[u] > 0) {
                const uint64_t *l = list + (slot * kG + u) * S;
                const bool f = t + u < own, all = before(l[len[u] - 1], q, f), none = !before(l[0], q, f);
                pos[u] = all ? len[u] : 0;
                need |= on && !all && !none;
            }
        }
        if (__any(need)) {   // (tiles of one order mostly stand apart)
#pragma unroll
            for (int u = 0; u < kG; u++) pos[u] = 0;
            for (int d = S; d; d >>= 1)
#pragma unroll
                for (int u = 0; u < kG; u++) {
                    const int p = pos[u] + d;
                    if (p <= len[u] && before(list[(slot * kG + u) * S + p - 1], q, t + u < own)) pos[u] = p;
                }
        }
#pragma unroll
        for (int u = 0; u < kG; u++) at += pos[u];
    }
    part[threadIdx.x] = at;
    __syncthreads();
    if (slot > 0 || !on) return;
    at = j;
    for (int k = 0; k < slots; k++) at += part[(k * groups + mine) * 64 + lane_id()];
    if (at > 0 && at % kBsPer == 0)
        split[at / kBsPer - 1] = Splitter{q, own, j * step + sample_phase(own, step)};
}

// Elements of tile u before a splitter.
template <int TILE>
__device__ inline int split_tile(const uint64_t *__restrict__ kin, int n, int u, const Splitter &s, int shift) {
    const int len = n - u * TILE < TILE ? n - u * TILE : TILE;
    if (u == s.tile) return s.pos;
    int p = 0;
    for (int d = TILE; d; d >>= 1)
        if (p + d <= len && before(kin[(size_t)u * TILE + p + d - 1] >> shift, s.q, u < s.tile)) p += d;
    return p;
}

// Bucket b of a set: pieces, gather, sort.
template <int TILE, int ITEMS>
__device__ __forceinline__ void bs_bucket(int n, int step, const uint64_t *__restrict__ kin,
                                          const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
                                          uint32_t *__restrict__ vout, int lo, const Splitter *__restrict__ split,
                                          int b) {
    __shared__ SortLds<ITEMS> S;
    __shared__ int from[kBsTiles], off[kBsTiles];
    __shared__ int scr[kMsWaves], low[kMsWaves];
    const int tid = threadIdx.x, w = tid >> 6, lane = lane_id(), shift = 8 * lo;
    const int tiles = (n + TILE - 1) / TILE;
    int samples = (tiles - 1) * (TILE / step) + sample_count(n, TILE, tiles - 1, step);
    const int buckets = samples > 0 ? (samples - 1) / kBsPer + 1 : 1;
    if (b >= buckets) return;
    // one tile per thread
    int l = 0, h = 0;
    if (tid < tiles) {
        // both ends searched side by side: a chain of log2(TILE) reads, not two
        const Splitter sl = split[b > 0 ? b - 1 : 0], sh = split[b < buckets - 1 ? b : 0];
        const int len = n - tid * TILE < TILE ? n - tid * TILE : TILE;
        const uint64_t *k = kin + (size_t)tid * TILE;
        for (int d = TILE; d; d >>= 1) {
            const uint64_t kl = k[l + d <= len ? l + d - 1 : 0] >> shift, kh = k[h + d <= len ? h + d - 1 : 0] >> shift;
            l += l + d <= len && before(kl, sl.q, tid < sl.tile) ? d : 0;
            h += h + d <= len && before(kh, sh.q, tid < sh.tile) ? d : 0;
        }
        l = b == 0 ? 0 : tid == sl.tile ? sl.pos : l;
        h = b == buckets - 1 ? len : tid == sh.tile ? sh.pos : h;
    }
    const int inc = wave_incl_scan(h - l);
    int lsum = l;
    for (int d = 32; d >= 1; d >>= 1) lsum += __shfl_xor(lsum, d, 64);
    if (lane == 63) { scr[w] = inc; low[w] = lsum; }
    __syncthreads();
    int at = inc - (h - l), size = 0, first = 0;
    for (int u = 0; u < kMsWaves; u++) {
        at += u < w ? scr[u] : 0;
        size += scr[u];
        first += low[u];
    }
    if (tid < tiles) { from[tid] = tid * TILE + l; off[tid] = at; }
    __syncthreads();
    // element i of the bucket: the last tile whose piece starts at or before it
    int top = 1;
    while (top < tiles) top <<= 1;
    auto source = [&](int i, int t) -> int { return from[t] + (i - off[t]); };
    if (size > ITEMS * kMsThreads) {
        // larger than the room: every key's place by searches in all tiles
        for (int i = tid; i < size; i += kMsThreads) {
            int t = 0;
            for (int d = top >> 1; d; d >>= 1)
                if (t + d < tiles && off[t + d] <= i) t += d;
            const int g = source(i, t);
            const uint64_t k = kin[g];
            const Splitter me{k >> shift, g / TILE, g % TILE};
            int r = 0;
            for (int u = 0; u < tiles; u++) r += split_tile<TILE>(kin, n, u, me, shift);
            kout[r] = k;
            vout[r] = vin[g];
        }
        return;
    }
    const int it = (size + kMsThreads - 1) / kMsThreads;
    const int base = w * (64 * it) + lane;
    uint64_t k[ITEMS];
    uint32_t v[ITEMS];
    int t[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) t[j] = 0;
    for (int d = top >> 1; d; d >>= 1)
#pragma unroll
        for (int j = 0; j < ITEMS; j++)
            if (j < it && t[j] + d < tiles && off[t[j] + d] <= base + j * 64) t[j] += d;
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        k[j] = 0ull;
        v[j] = 0u;
        if (j < it && base + j * 64 < size) {
            const int g = source(base + j * 64, t[j]);
            k[j] = kin[g];
            v[j] = vin[g];
        }
    }
    lds_sort<ITEMS>(S, k, v, it, size, lo);
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const int p = base + j * 64;
        if (j < it && p < size) { kout[first + p] = k[j]; vout[first + p] = v[j]; }
    }
}

// The samples' step for n keys (64 steps: a bucket's average).
static int bs_step(int64_t n) { return n <= 262144 ? 16 : n <= 524288 ? 32 : 64; }

template <int TILE>
__global__ __launch_bounds__(kMsThreads) void k_bs_split(int n, int step, const uint64_t *__restrict__ samp,
                                                         Splitter *split) {
    bs_split<TILE>(n, step, samp, split, blockIdx.x);
}

template <int TILE, int ITEMS>
__global__ __launch_bounds__(kMsThreads) void k_bs_bucket(int n, int step, const uint64_t *__restrict__ kin,
                                                          const uint32_t *__restrict__ vin,
                                                          uint64_t *__restrict__ kout, uint32_t *__restrict__ vout,
                                                          int lo, const Splitter *__restrict__ split) {
    bs_bucket<TILE, ITEMS>(n, step, kin, vin, kout, vout, lo, split, blockIdx.x);
}

template <int TILE>
__global__ __launch_bounds__(kMsThreads) void k_ms_tile(int n, const uint64_t *__restrict__ kin,
                                                        const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
                                                        uint32_t *__restrict__ vout, int lo,
                                                        uint64_t *__restrict__ samp, int step) {
    ms_tile<TILE>(n, kin, vin, kout, vout, lo, blockIdx.x, samp, step);
}

// The same for a set whose keys all fit in LDS (kMsTiny): 1024 threads place
// 256 keys, searching copies there instead of through L2 (sort phase 10,000
// particles 29.5 -> 26.4 us, 15,000 30.0 -> 26.6).
__global__ __launch_bounds__(kMsThreads) void k_ms_merge_lds(int n, const uint64_t *__restrict__ kin,
                                                             const uint32_t *__restrict__ vin,
                                                             uint64_t *__restrict__ kout,
                                                             uint32_t *__restrict__ vout, int lo) {
    __shared__ uint64_t keys[kMsTiny];
    constexpr int kRows = kMsTiny / kMsThreads;
    uint64_t row[kRows];   // every load before the first store
#pragma unroll
    for (int u = 0; u < kRows; u++) {
        const int i = u * kMsThreads + (int)threadIdx.x;
        row[u] = i < n ? kin[i] : 0ull;
    }
#pragma unroll
    for (int u = 0; u < kRows; u++) keys[u * kMsThreads + threadIdx.x] = row[u];
    __syncthreads();
    ms_merge<kMsTiny0>(n, keys, vin, kout, vout, lo, blockIdx.x * (kMsThreads / kMsLanes) + threadIdx.x / kMsLanes);
}

template <int TILE>
__global__ __launch_bounds__(256) void k_ms_merge(int n, const uint64_t *__restrict__ kin,
                                                  const uint32_t *__restrict__ vin, uint64_t *__restrict__ kout,
                                                  uint32_t *__restrict__ vout, int lo) {
    ms_merge<TILE>(n, kin, vin, kout, vout, lo, blockIdx.x * kMsPer + threadIdx.x / kMsLanes);
}

// Batched sort of several contexts (a serving round): job j's tiles are the
// workgroups [tile0, tile0 + nblk) of one launch per kernel and pass, found
// by binary search; each job keeps its own buffers, so its result is that of
// its own sort.
struct SortJob {
    int n, nblk, tile0, pad;
    uint64_t *key, *key_alt;
    uint32_t *idx, *idx_alt;
    uint32_t *hist, *dtotal;
    uint64_t *samp;   // key2, which is written after the sort: samples, then splitters
};

__device__ inline int find_sort_job(const SortJob *jobs, int nj, int b) {
    int lo = 0, hi = nj - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].tile0 <= b) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(256) void k_rsb_hist(const SortJob *jobs, int nj, int pass) {
    const SortJob &J = jobs[find_sort_job(jobs, nj, blockIdx.x)];
    rs_hist_tile(J.n, (pass & 1) ? J.key_alt : J.key, 8 * pass, J.hist, J.nblk, (int)blockIdx.x - J.tile0);
}

template <int TILE>
__global__ __launch_bounds__(kMsThreads) void k_msb_tile(const SortJob *jobs, int nj, int lo, int step) {
    const SortJob &J = jobs[find_sort_job(jobs, nj, blockIdx.x)];
    ms_tile<TILE>(J.n, J.key, J.idx, J.key_alt, J.idx_alt, lo, (int)blockIdx.x - J.tile0, J.samp, step);
}

// (64 samples a tile in a batch: one bucket's worth)
template <int TILE>
__global__ __launch_bounds__(kMsThreads) void k_bsb_split(const SortJob *jobs, int nj) {
    const SortJob &J = jobs[find_sort_job(jobs, nj, blockIdx.x)];
    bs_split<TILE>(J.n, TILE / kBsPer, J.samp, (Splitter *)(J.samp + (size_t)J.nblk * kBsPer),
                   (int)blockIdx.x - J.tile0);
}

template <int TILE, int ITEMS>
__global__ __launch_bounds__(kMsThreads) void k_bsb_bucket(const SortJob *jobs, int nj, int lo) {
    const SortJob &J = jobs[find_sort_job(jobs, nj, blockIdx.x)];
    bs_bucket<TILE, ITEMS>(J.n, TILE / kBsPer, J.key_alt, J.idx_alt, J.key, J.idx, lo,
                           (const Splitter *)(J.samp + (size_t)J.nblk * kBsPer), (int)blockIdx.x - J.tile0);
}

template <int TILE>
__global__ __launch_bounds__(256) void k_msb_merge(const SortJob *jobs, int nj, int lo) {
    constexpr int kPer = TILE / kMsPer;   // workgroups per tile
    const SortJob &J = jobs[find_sort_job(jobs, nj, blockIdx.x / kPer)];
    const int b = (int)blockIdx.x - J.tile0 * kPer;
    if (b * kMsPer < J.n)
        ms_merge<TILE>(J.n, J.key_alt, J.idx_alt, J.key, J.idx, lo, b * kMsPer + (int)threadIdx.x / kMsLanes);
}

__global__ __launch_bounds__(256) void k_rsb_scan(const SortJob *jobs) {
    const SortJob &J = jobs[blockIdx.x >> 8];
    rs_scan_digit(J.nblk, J.hist, J.dtotal, blockIdx.x & 255);
}

__global__ __launch_bounds__(256) void k_rsb_scatter(const SortJob *jobs, int nj, int pass) {
    const SortJob &J = jobs[find_sort_job(jobs, nj, blockIdx.x)];
    const bool odd = pass & 1;
    rs_scatter_tile<false>(J.n, odd ? J.key_alt : J.key, odd ? J.idx_alt : J.idx, odd ? J.key : J.key_alt,
                           odd ? J.idx : J.idx_alt, 8 * pass, J.hist, J.dtotal, J.nblk, (int)blockIdx.x - J.tile0);
}

// ------------------------------------------------------------ after sort

// Longest run of particles sharing the sorted bits that k_tie_rank orders.
constexpr int kTieRankMax = 1024;

// First and last particle of the run sharing k[i] >> shift (galloping).
__device__ inline int word_run_first(const uint64_t *k, int i, int shift = 0) {
    const uint64_t pi = k[i] >> shift;
    int hi = i, lo = -1;
    for (int step = 1;; step <<= 1) {
        const int probe = i - step;
        if (probe < 0) break;
        if ((k[probe] >> shift) != pi) { lo = probe; break; }
        hi = probe;
        if (step > (1 << 29)) break;
    }
    while (hi - lo > 1) {
        const int mid = lo + ((hi - lo) >> 1);
        if ((k[mid] >> shift) == pi) hi = mid; else lo = mid;
    }
    return hi;
}

__device__ inline int word_run_last(const uint64_t *k, int i, int nin, int shift = 0) {
    const uint64_t pi = k[i] >> shift;
    int lo = i, hi = nin;
    for (int step = 1;; step <<= 1) {
        const int probe = i + step;
        if (probe >= nin) break;
        if ((k[probe] >> shift) != pi) { hi = probe; break; }
        lo = probe;
        if (step > (1 << 29)) break;
    }
    while (hi - lo > 1) {
        const int mid = lo + ((hi - lo) >> 1);
        if ((k[mid] >> shift) == pi) lo = mid; else hi = mid;
    }
    return lo;
}

// The particles in the root cube (sorted before the others, whose key is
// kOut) -> ds->nin.  Runs of particles sharing the sorted bits of word 0
// (key >> shift) are ordered by k_tie_rank; a particle whose whole word 0
// another particle of its run has gets its levels 22..42 (word 1) here.
// kOut shares no prefix with a key in the cube (bit 63 is clear in those),
// so runs stay below nin.
__global__ __launch_bounds__(256) void k_tie_key2(int n, const uint64_t *key, const uint32_t *idx,
                                                  const double *x, const double *y, const double *z,
                                                  DevState *ds, uint64_t *key2, uint8_t *gapl, int shift) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint64_t ki = key[i];
    const bool in = ki != kOut;
    if (in && (i + 1 == n || key[i + 1] == kOut)) ds->nin = i + 1;
    if (i == 0 && !in) ds->nin = 0;
    if (!in) return;
    const uint64_t pi = ki >> shift;
    const bool run = (i > 0 && (key[i - 1] >> shift) == pi) || (i + 1 < n && (key[i + 1] >> shift) == pi);
    if (!run) return;   // k_tie_rank reads word 1 of run members only
    bool tie = true;
    if (shift > 0) {
        // short runs: is the whole key shared?  (a run too long for the
        // ranking sends the build back to a full sort)
        tie = false;
        const int s = word_run_first(key, i, shift), e = word_run_last(key, i, n, shift);
        if (e - s + 1 <= kTieRankMax)
            for (int j = s; j <= e && !tie; j++) tie = j != i && key[j] == ki;
    }
    if (!tie) { key2[i] = 0ull; return; }
    double R = __longlong_as_double((long long)ds->Rbits);
    uint32_t q = idx[i];
    uint64_t a, b;
    int g;
    core::octant_path(x[q], y[q], z[q], R, 42, &a, &b, &g);
    key2[i] = b;
    if (gapl[q] == 0 && g > 0) gapl[q] = (uint8_t)(g > 254 ? 254 : g);
}

// Runs of particles sharing key >> shift (the radix-sorted bits) take their
// order by (word 0, word 1, caller index): the reference inserts particles
// of one cell in array order (Tree.cpp:44-48) whatever resident order they
// were sorted from.  Each particle of a run of k counts the members before it
// (k steps per thread), and everything goes to the output buffers: word 0 to
// w0, word 1 to w1, the sort permutation to ord (particles outside runs keep
// their place).  Runs longer than kTieRankMax are left in order and flagged
// in ds->tie_big: the build then sorts every byte of word 0 again (shift >
// 0) or refines them with the general segmented sort (refine_ties).
__global__ __launch_bounds__(256) void k_tie_rank(int n, const uint64_t *key, const uint64_t *key2,
                                                  const uint32_t *idx, const uint32_t *rid, DevState *ds,
                                                  uint64_t *w0, uint64_t *w1, uint32_t *ord, int shift) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int nin = ds->nin;
    const uint64_t k0 = key[i];
    if (i >= nin) { ord[i] = idx[i]; w0[i] = k0; return; }
    const uint64_t p0 = k0 >> shift;
    const bool run = (i > 0 && (key[i - 1] >> shift) == p0) || (i + 1 < nin && (key[i + 1] >> shift) == p0);
    if (!run) { ord[i] = idx[i]; w0[i] = k0; w1[i] = 0ull; return; }
    const int s = word_run_first(key, i, shift), e = word_run_last(key, i, nin, shift);
    if (i == s) atomicMax(&ds->max_prefix_run, e - s + 1);
    if (e - s + 1 > kTieRankMax) {
        ord[i] = idx[i];
        w0[i] = k0;
        w1[i] = key2[i];
        if (i == s) ds->tie_big = 1;
        return;
    }
    const uint64_t ki = key2[i];
    const uint32_t ci = rid[idx[i]];
    int rank = 0;
    for (int j = s; j <= e; j++) {
        const uint64_t kj0 = key[j];
        if (kj0 < k0) {
            rank++;
        } else if (kj0 == k0) {
            const uint64_t kj = key2[j];
            rank += (kj < ki || (kj == ki && rid[idx[j]] < ci)) ? 1 : 0;
        }
    }
    ord[s + rank] = idx[i];
    w0[s + rank] = k0;
    w1[s + rank] = ki;
}

// The whole particle state moves into the new key order: out[k] = in[idx[k]].
// Particles move little between steps, so idx is close to the identity and
// the reads stay nearly coalesced.
struct StateSet {
    double *d[kStateD];
    uint8_t *type, *active;
    uint32_t *rid;
};

// Output slots in XCD ranges: neighbouring slots gather from neighbouring
// source lines, which then share one L2.
// skip_acc: fields kAccField .. kAccField + 2 (the accelerations) are left
// out, for a build whose force phase writes every one of them.  zero_gas_h:
// field kHField (h) becomes 0 for gas, for a build whose density phase
// follows (it starts so, Tree.cpp:121-130).
// PARTS: the fields shared by so many workgroups of the grid's second
// dimension.  Up to 131,072 particles the chip is not full and a thread's
// nineteen gathers are what it waits for: five parts of four fields take 4.8
// us against 7.7 at 10,000, 5.7 against 8.4 at 33,333, 6.5 against 8.3 at
// 100,000; 10.1 against 10.3 at 150,000, 14.3 against 13.8 at 200,000, and
// more above (1,000,000: 60 against 52).
constexpr int kAccField = 9;
constexpr int kHField = 12;
constexpr int kPermuteParts = 5, kPermuteSplit = 131072;

template <int PARTS>
__global__ __launch_bounds__(256) void k_permute(int n, const uint32_t *__restrict__ idx, StateSet in, StateSet out,
                                                 int skip_acc, int zero_gas_h) {
    int k = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (k >= n) return;
    uint32_t q = idx[k];
    const uint8_t ty = in.type[q];
    constexpr int kPer = (kStateD + PARTS - 1) / PARTS;
    const int j0 = PARTS > 1 ? (int)blockIdx.y * kPer : 0;
#pragma unroll
    for (int u = 0; u < kPer; u++) {
        const int j = j0 + u;
        if (j >= kStateD || (skip_acc && j >= kAccField && j < kAccField + 3)) continue;
        out.d[j][k] = (j == kHField && zero_gas_h && ty == 2) ? 0.0 : in.d[j][q];
    }
    if (PARTS > 1 && blockIdx.y > 0) return;
    out.type[k] = ty;
    out.active[k] = in.active[q];
    out.rid[k] = in.rid[q];
}

__global__ __launch_bounds__(256) void k_inverse(int n, const uint32_t *rid, int32_t *inv) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r < n) inv[rid[r]] = r;
}

// lv[i] = L[i] + 1 (0 .. 127; L: the levels particles i and i + 1 share, -1
// after the last one inside) and c[i] = max(0, L[i] - L[i-1]), over the key
// words of this build (nw of them) and the positions in key order (runs at
// one position are buckets).  A distinct pair that agrees on every word sets
// ds->tie_deep: the build refines it with deeper words (refine_ties), or
// fails past kDeepest levels.
// One particle per thread, a 1024-particle scan tile per workgroup (four per
// thread of 256 waited for each one's loads in turn: 7.5 us at 10,000
// particles, now 4.6); the tile's sum of c goes to bsum for k_scan_apply, the
// least lv of the tile (0 past the last particle) to lmin for the cell
// searches.
constexpr int kLevTile = 1024;

__global__ __launch_bounds__(kLevTile) void k_lcp(int n, core::KeyWords kw, int nw, core::Pos pos, DevState *ds,
                                                  int parallel_root, uint8_t *lv, uint8_t *lmin, int32_t *c,
                                                  int32_t *bsum) {
    __shared__ int level[kLevTile], wsum[kLevTile / 64], wmin[kLevTile / 64];
    const int nin = ds->nin;
    const bool proot = parallel_root != 0, splits = proot && nin < n;
    const int i = blockIdx.x * kLevTile + threadIdx.x;
    int li = -1, v = 0;
    if (i < nin) {
        li = core::pair_lcp(kw, pos, i, nin, proot, splits);
        // a coincident pair's level is its bucket's (pair_lcp), whatever the key words say
        const bool coincident = i + 1 < nin && core::same_pos(pos, i, i + 1);
        if (coincident) ds->any_bucket = 1;
        if (i + 1 < nin && li >= 21 * nw && !coincident) ds->tie_deep = 1;
        if (li > core::kDeepest) { li = core::kDeepest; ds->tie_deep = 1; }
    }
    lv[i] = (uint8_t)(li + 1);
    level[threadIdx.x] = li;
    __syncthreads();
    if (i < nin) {
        int lp = -1;
        if (threadIdx.x > 0) lp = level[threadIdx.x - 1];
        else if (i > 0) lp = core::pair_lcp(kw, pos, i - 1, nin, proot, splits);
        if (lp > core::kDeepest) lp = core::kDeepest;
        v = li - lp > 0 ? li - lp : 0;
        c[i] = v;
    }
    int least = li + 1;
    for (int d = 32; d >= 1; d >>= 1) {
        const int t = __shfl_xor(least, d, 64);
        least = t < least ? t : least;
        v += __shfl_xor(v, d, 64);
    }
    if (lane_id() == 0) { wsum[threadIdx.x >> 6] = v; wmin[threadIdx.x >> 6] = least; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kLevTile / 64; w++) {
            v += wsum[w];
            least = wmin[w] < least ? wmin[w] : least;
        }
        bsum[blockIdx.x] = v;
        lmin[blockIdx.x] = (uint8_t)least;
    }
}

// The exclusive scan of c into base over tiles of 1024 (256 threads x 4):
// each tile forms its own offset from the tile sums k_lcp left; tile 0 also
// records the node counts.
__global__ __launch_bounds__(256) void k_scan_apply(const int32_t *c, const int32_t *bsum, DevState *ds,
                                                    int parallel_root, int64_t node_cap, int32_t *base) {
    __shared__ int scr[4];
    int nin = ds->nin;
    int b0 = blockIdx.x * 1024 + threadIdx.x * 4;
    int v[4];
    int s = 0;
    for (int k = 0; k < 4; k++) { v[k] = (b0 + k < nin) ? c[b0 + k] : 0; s += v[k]; }
    int tot;
    const int pre = tile_offset(bsum, (int)gridDim.x, (int)blockIdx.x, scr, &tot);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        int n_int = (nin == 0) ? (parallel_root ? 1 : 0) : tot;
        ds->n_int = n_int;
        ds->n_nodes = n_int + nin;
        if ((int64_t)n_int + nin > node_cap) ds->err = 1;
    }
    int ex = block256_excl_scan(s, scr, nullptr) + pre;
    for (int k = 0; k < 4; k++) {
        if (b0 + k <= nin) base[b0 + k] = ex;
        ex += v[k];
    }
}

// ------------------------------------------------------------ nodes
// The tree from the levels alone.  A particle starts c[i] internal nodes, of
// levels L[i-1] + 1 .. L[i], then its leaf; the internal nodes, numbered q =
// 0 .. n_int - 1 in pre-order, are those of particle i for base[i] <= q <
// base[i] + c[i] (k_make_leaf lists own[q] = i), and node q of particle i
// sits at pre-order index i + q.  The level-l node from particle i on ends
// with the first j >= i whose L[j] < l, and every j before that with L[j] ==
// l ends one child: the next starts at particle j + 1, as its first node.  So
// the end, the children and their ranks come out of one search for levels <=
// l, with no look at the keys.  (Members of a bucket, whose L is the bucket's
// level, come out as its children.)
struct NodeArrays {
    int32_t *first, *count, *parent, *pidx, *nchild, *rank;
    int8_t *level;
};

// The bytes of x below t (bytes 0 .. 127, t 1 .. 128 in every byte of t4), as
// 4 bits scaled by 128, shifted up by 4 with HI.
template <bool HI>
__device__ inline unsigned below4(unsigned x, unsigned t4, unsigned acc) {
    const unsigned less = ~((x | 0x80808080u) - t4) & 0x80808080u;
    return (unsigned)__builtin_amdgcn_udot4(less, HI ? 0x80402010u : 0x08040201u, acc, false);
}

typedef unsigned levels16 __attribute__((ext_vector_type(4), aligned(4)));

// Which of 16 bytes are below t, 16 bits.
__device__ inline unsigned below16(const levels16 &x, unsigned t4) {
    const unsigned a = below4<true>(x[1], t4, below4<false>(x[0], t4, 0u));
    const unsigned b = below4<true>(x[3], t4, below4<false>(x[2], t4, 0u));
    return a >> 7 | b << 1;
}

// Which of the 64 levels from particle i on are below t; x: the 68 bytes from
// i & ~3 on.
__device__ inline unsigned long long below64(const levels16 (&x)[4], unsigned x4, int sh, unsigned t4) {
    unsigned long long m = 0ull;
#pragma unroll
    for (int k = 0; k < 4; k++) m |= (unsigned long long)below16(x[k], t4) << (16 * k);
    const unsigned long long up = below4<false>(x4, t4, 0u) >> 7;
    return sh ? m >> sh | up << (64 - sh) : m;
}

// The boundaries among the 16 levels of each lane (bit b of le: the particle
// after p0 + b starts a child), as children run + 1, run + 2, .. of node nd;
// returns their number.
__device__ inline int emit_children(unsigned le, int p0, int nd, int run, const int32_t *base, const NodeArrays &o) {
    const unsigned long long any = __ballot(le != 0);
    int r = run + __popcll(any & lanes_below()), total = __popcll(any);
    if (__ballot((le & (le - 1)) != 0)) {   // more than one in some lane
        const int k = __popc(le);
        const int inc = wave_incl_scan(k);
        r = run + inc - k;
        total = __shfl(inc, 63, 64);
    }
    while (le) {
        const int p = p0 + __builtin_ctz(le) + 1;
        le &= le - 1;
        const int ch = p + base[p];
        o.parent[ch] = nd;
        o.rank[ch] = ++r;
    }
    return total;
}

// 1024 levels from s on (a multiple of 16) for a node: every boundary from i
// on in them, up to the node's end if that is here (returned; -1: the node
// goes on).
__device__ inline int scan_levels(const uint8_t *lv, int s, int i, unsigned lt4, unsigned le4, int nd, int *run,
                                const int32_t *base, const NodeArrays &o) {
    const int p0 = s + lane_id() * 16;
    const levels16 x = *(const levels16 *)(lv + p0);
    const int cut = i - p0;
    const unsigned from = cut <= 0 ? 0xffffu : cut >= 16 ? 0u : 0xffffu << cut & 0xffffu;
    const unsigned lt = below16(x, lt4) & from;
    unsigned le = below16(x, le4) & from;
    const unsigned long long f = __ballot(lt != 0);
    int end = -1;
    if (f) {
        const int fl = __builtin_ctzll(f);
        const int at = __builtin_ctz(__shfl(lt, fl, 64));
        end = s + fl * 16 + at;
        le = lane_id() < fl ? le : lane_id() == fl ? le & ((1u << at) - 1) : 0u;
    }
    if (__ballot(le != 0)) *run += emit_children(le, p0, nd, *run, base, o);
    return end;
}

// One thread per internal node.  A node whose end is among the 64 levels from
// its first particle on (and that has at most 8 children) is found by its
// thread, in one read; the others, a few in a hundred, are listed and shared by
// the workgroup's waves: the 1024 levels from the first particle on, the rest
// of the tile they end in, then the tiles' least levels, then the tiles that hold a child's end, a read each.  tsum
// (zeroed by k_make_leaf) gets the children of every 1024 nodes for
// k_iscan_apply.
// Galloping searches over the keys for each node's end and its parent's
// start, then a pass that followed the children by their skip links, were
// chains of 10 to 50 dependent reads: make_leaf, make_internal and
// child_count took 14 + 17 + 11 us at 10,000 particles and 37 + 39 + 17 us at
// 1,000,000; now make_leaf and make_internal 4.4 + 9.5 and 15 + 30.
template <int PER>
__global__ __launch_bounds__(256) void k_make_internal(int nin, int n_int, const uint8_t *lv, const uint8_t *lmin,
                                                       const int32_t *base, const int32_t *own, NodeArrays o,
                                                       int32_t *tsum) {
    __shared__ int w_i[PER], w_l[PER], w_nd[PER], n_wide;
    if (threadIdx.x == 0) n_wide = 0;
    __syncthreads();
    const int q = xcd_block(blockIdx.x, gridDim.x) * PER + threadIdx.x;
    const bool have = (int)threadIdx.x < PER && q < n_int;
    int nch = 0, nd = 0;
    if (have) {
        const int i = own[q];
        const int l = (i > 0 ? (int)lv[i - 1] : 0) + (q - base[i]);
        nd = i + q;
        levels16 x[4];
        const uint8_t *w = lv + (i & ~3);
#pragma unroll
        for (int k = 0; k < 4; k++) x[k] = *(const levels16 *)(w + 16 * k);
        const unsigned x4 = *(const unsigned *)(w + 64);
        const unsigned long long lt = below64(x, x4, i & 3, (unsigned)(l + 1) * 0x01010101u);
        unsigned long long le = below64(x, x4, i & 3, (unsigned)(l + 2) * 0x01010101u);
        o.first[nd] = i;
        o.pidx[nd] = -1;
        o.level[nd] = (int8_t)l;
        if (nd == 0) o.parent[0] = -1;
        o.parent[nd + 1] = nd;
        o.rank[nd + 1] = 0;
        // a tree of one particle under a root that always splits has no level below the root's
        int e = lt ? __builtin_ctzll(lt) : 64;
        e = i + e > nin - 1 ? nin - 1 - i : e;
        le &= e < 64 ? (1ull << e) - 1 : ~0ull;
        const int more = __popcll(le);
        if (e < 64 && more <= 7) {
            o.count[nd] = e + 1;
            o.nchild[nd] = nch = more + 1;
            int p[7], b[7];
#pragma unroll
            for (int k = 0; k < 7; k++) {
                p[k] = le ? i + __builtin_ctzll(le) + 1 : i;
                le &= le - 1;
            }
#pragma unroll
            for (int k = 0; k < 7; k++) b[k] = base[p[k]];
#pragma unroll
            for (int k = 0; k < 7; k++)
                if (k < more) {
                    o.parent[p[k] + b[k]] = nd;
                    o.rank[p[k] + b[k]] = k + 1;
                }
        } else {
            const int at = atomicAdd(&n_wide, 1);
            w_i[at] = i;
            w_l[at] = l;
            w_nd[at] = nd;
        }
    }
    // the children of the threads' own nodes (1 .. 8 each), by tile of nodes
    unsigned long long left = __ballot(nch > 0);
    while (left) {
        const int f = __builtin_ctzll(left);
        const int t = __shfl(nd >> 10, f, 64);
        const bool in = nch > 0 && (nd >> 10) == t;
        int s = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) s += __popcll(__ballot(in && (nch >> k & 1))) << k;
        if (lane_id() == f) atomicAdd(&tsum[t], s);
        left &= ~__ballot(in);
    }
    __syncthreads();
    const int nw = n_wide;
    for (int k = threadIdx.x >> 6; k < nw; k += 4) {
        const int i = w_i[k], l = w_l[k], node = w_nd[k];
        const unsigned lt4 = (unsigned)(l + 1) * 0x01010101u, le4 = (unsigned)(l + 2) * 0x01010101u;
        int run = 0;
        const int s = i & ~15, tile = (s + 2 * kLevTile - 1) / kLevTile;   // the first tile all past s + 1023
        int end = scan_levels(lv, s, i, lt4, le4, node, &run, base, o);
        if (end < 0 && s % kLevTile)
            end = scan_levels(lv, (tile - 1) * kLevTile, s + kLevTile, lt4, le4, node, &run, base, o);
        for (int t0 = tile & ~15, from = tile; end < 0; t0 += kLevTile, from = t0) {
            // the tile of particle nin - 1 holds a level below every l, so
            // the search ends there at the latest
            const int p0 = t0 + lane_id() * 16;
            const levels16 x = *(const levels16 *)(lmin + p0);
            const int cut = from - p0;
            const unsigned in = cut <= 0 ? 0xffffu : cut >= 16 ? 0u : 0xffffu << cut & 0xffffu;
            // tiles with a child's end or the node's, in order
            unsigned le = below16(x, le4) & in;
            unsigned long long b = __ballot(le != 0);
            while (b && end < 0) {
                const int f = __builtin_ctzll(b);
                b &= b - 1;
                unsigned m = __shfl(le, f, 64);
                while (m && end < 0) {
                    end = scan_levels(lv, (t0 + f * 16 + __builtin_ctz(m)) * kLevTile, i, lt4, le4, node, &run, base, o);
                    m &= m - 1;
                }
            }
        }
        if (lane_id() == 0) {
            o.count[node] = end - i + 1;
            o.nchild[node] = run + 1;
            atomicAdd(&tsum[node >> 10], run + 1);
        }
    }
}

__global__ __launch_bounds__(256) void k_make_root_only(NodeArrays o, int32_t *tsum) {
    if (threadIdx.x == 0) {
        o.first[0] = 0; o.count[0] = 0; o.parent[0] = -1; o.pidx[0] = -1; o.level[0] = 0;
        o.nchild[0] = 0; o.rank[0] = 0;
        tsum[0] = 0;
    }
}

// The leaves (one per particle), the list of the particles that start the
// internal nodes, and per tile of 1024 particles the deepest leaf level and
// the number of gaps (part: level | gaps << 8).  It needs nothing of the host,
// so it runs while the host waits for the counts; when the nodes are more
// than the room (ds->err) it writes nothing, and the host launches it again
// after making room.
__global__ __launch_bounds__(kLevTile) void k_make_leaf(const DevState *ds, const uint8_t *lv, const int32_t *base,
                                                        const int32_t *c, NodeArrays o, const uint32_t *idx,
                                                        const uint8_t *gapl, int32_t *own, int32_t *tsum,
                                                        int32_t *part) {
    __shared__ int wl[kLevTile / 64], wg[kLevTile / 64];
    if (ds->err) return;
    const int i = blockIdx.x * kLevTile + threadIdx.x;
    for (int k = i; k <= ds->n_nodes / 1024; k += gridDim.x * kLevTile) tsum[k] = 0;
    int deep = 0, gp = 0;
    if (i < ds->nin) {
        const int a = i > 0 ? lv[i - 1] : 0, b = lv[i];
        const int li = a > b ? a : b;   // one level below the deeper neighbour pair
        const int b0 = base[i], ci = c[i];
        const int g = gapl[idx[i]];
        const int nd = i + b0 + ci;
        o.first[nd] = i;
        o.count[nd] = 1;
        o.pidx[nd] = i;
        o.level[nd] = (int8_t)li;
        o.nchild[nd] = 0;
        if (nd == 0) o.parent[0] = -1;
        // particle i starts internal nodes base[i] .. base[i] + c[i] - 1
        for (int u = 0; u < ci; u++) own[b0 + u] = i;
        deep = li;
        gp = (g > 0 && g <= li) ? 1 : 0;
    }
    for (int d = 32; d >= 1; d >>= 1) {
        const int t = __shfl_xor(deep, d, 64);
        deep = t > deep ? t : deep;
        gp += __shfl_xor(gp, d, 64);
    }
    if (lane_id() == 0) { wl[threadIdx.x >> 6] = deep; wg[threadIdx.x >> 6] = gp; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kLevTile / 64; w++) { deep = wl[w] > deep ? wl[w] : deep; gp += wg[w]; }
        part[blockIdx.x] = deep | gp << 8;
    }
}

// Deepest leaf level and gap count from make_leaf's per-tile partials
// (one workgroup of 256; run by the first workgroup of k_iscan_apply).
__device__ inline void leaf_fold(int nb, const int32_t *part, DevState *ds) {
    __shared__ int wl[4], wg[4];
    int lv = 0, gp = 0;
    for (int k = threadIdx.x; k < nb; k += 256) {
        const int p = part[k];
        lv = (p & 0xff) > lv ? p & 0xff : lv;
        gp += p >> 8;
    }
    for (int o = 32; o >= 1; o >>= 1) {
        const int q = __shfl_xor(lv, o, 64);
        lv = q > lv ? q : lv;
        gp += __shfl_xor(gp, o, 64);
    }
    if (lane_id() == 0) { wl[threadIdx.x >> 6] = lv; wg[threadIdx.x >> 6] = gp; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; w++) { lv = wl[w] > lv ? wl[w] : lv; gp += wg[w]; }
        ds->max_level = lv;
        // stack growth bound: at most 7 blocks per level below
        ds->walk_depth = 7 * (lv + 3);
        ds->gap = (unsigned long long)gp;
    }
}

// ------------------------------------------------------------ moments
// Node sums (mass, mass-weighted position, gas mass, gas-mass-weighted
// velocity) straight from each internal node's particle range in key order,
// in a fixed order that depends on the range alone, so they are
// deterministic and round relative to the node's own terms wherever the
// rest of the system lies.  No node waits for another: a bottom-up pass
// would chain the deepest leaf's latency through every level.
//
// k_tile_sums forms the sums of aligned blocks of kBlk1 = 64 particles (a
// butterfly over one wave) and of kBlk2 = 4096 (a butterfly over its 64
// blocks).  A node of up to kSumSmall particles is summed by one lane in
// index order from particles its workgroup staged in LDS; a larger one by a
// wave, over the greedy ascending cover of its range by particles, 64-blocks
// and 4096-blocks (lane j taking pieces j, j + 64, ...; then a butterfly),
// the parallel root adding the particles outside its cube (Node.cpp:477-499)
// as further pieces.
constexpr int kSumSmall = 32;
constexpr int kBlk1 = 64;
constexpr int kBlk2 = 4096;

struct PVals {
    const double *sx, *sy, *sz, *sm, *svx, *svy, *svz;
    const uint8_t *stype;
};

// Butterflies over the wave (lane distances 32, 16, .. 1) of several sums at
// once, in halving form: at each distance a pair of lanes exchanges half of
// its sums and each adds the other half, so that a sum takes one exchange in
// all instead of six per lane.  Every sum adds the same terms in the same
// order as a plain butterfly.  The exchanges stay on the vector unit: the 96
// LDS permutes per eight sums of the plain form were what bounded the node
// sums (k_tile_sums at 10,000 particles, whose three workgroups sit on three
// CUs: 21.5 -> 5.5 us; 1,000,000: 29 -> 15 us).
template <int CTRL>
__device__ inline double dpp_f64(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)u, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
}
__device__ inline double lane_xor8(double v) { return dpp_f64<0x128>(v); }                 // row_ror:8
__device__ inline double lane_xor4(double v) { return dpp_f64<0x1b>(dpp_f64<0x141>(v)); }   // ^ 7, then ^ 3
__device__ inline double lane_xor2(double v) { return dpp_f64<0x4e>(v); }
__device__ inline double lane_xor1(double v) { return dpp_f64<0xb1>(v); }

// Lanes with bit 5 (4) clear get a's sum over the lane pair at distance 32
// (16), the others b's.
template <int D>
__device__ inline double halve_swap(double a, double b) {
    const unsigned long long ua = __builtin_bit_cast(unsigned long long, a);
    const unsigned long long ub = __builtin_bit_cast(unsigned long long, b);
    unsigned long long x, y;
    if (D == 32) {
        auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
        auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
        x = (unsigned long long)hi[0] << 32 | lo[0];
        y = (unsigned long long)hi[1] << 32 | lo[1];
    } else {
        auto lo = __builtin_amdgcn_permlane16_swap((unsigned)ua, (unsigned)ub, false, false);
        auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
        x = (unsigned long long)hi[0] << 32 | lo[0];
        y = (unsigned long long)hi[1] << 32 | lo[1];
    }
    return __builtin_bit_cast(double, x) + __builtin_bit_cast(double, y);
}
__device__ inline double halve8(double a, double b) {
    const bool up = (lane_id() & 8) != 0;
    return (up ? b : a) + lane_xor8(up ? a : b);
}
__device__ inline double halve4(double a, double b) {
    const bool up = (lane_id() & 4) != 0;
    return (up ? b : a) + lane_xor4(up ? a : b);
}
__device__ inline double halve2(double a, double b) {
    const bool up = (lane_id() & 2) != 0;
    return (up ? b : a) + lane_xor2(up ? a : b);
}

// Eight sums over the wave: lane l gets sum l >> 3.
__device__ inline double wave_sums8(const double (&v)[8]) {
    double r[4];
#pragma unroll
    for (int j = 0; j < 4; j++) r[j] = halve_swap<32>(v[j], v[j + 4]);
    double s = halve8(halve_swap<16>(r[0], r[2]), halve_swap<16>(r[1], r[3]));
    s += lane_xor4(s);
    s += lane_xor2(s);
    s += lane_xor1(s);
    return s;
}

// Thirty-two sums over the wave: lane l gets sum l >> 1.
__device__ inline double wave_sums32(const double (&v)[32]) {
    double r[16];
#pragma unroll
    for (int j = 0; j < 16; j++) r[j] = halve_swap<32>(v[j], v[j + 16]);
#pragma unroll
    for (int j = 0; j < 8; j++) r[j] = halve_swap<16>(r[j], r[j + 8]);
#pragma unroll
    for (int j = 0; j < 4; j++) r[j] = halve8(r[j], r[j + 4]);
    double s = halve2(halve4(r[0], r[2]), halve4(r[1], r[3]));
    s += lane_xor1(s);
    return s;
}

// One workgroup of 16 waves per 4096 particles: wave w forms blocks 4 w ..
// 4 w + 3 of 64, then wave 0 the 4096-block from the 64.  Blocks past nin
// hold zeros.  The grid covers all n particles: the launch does not wait
// for the host to learn nin.
__global__ __launch_bounds__(1024) void k_tile_sums(const DevState *ds, PVals v, NodeSums *blk1, NodeSums *blk2) {
    static_assert(sizeof(NodeSums) == 64, "a block's sums are written as eight doubles");
    __shared__ double sb[8][64 + 1];
    const int nin = ds->nin;
    const int w = threadIdx.x >> 6, lane = lane_id();
    const int b0 = blockIdx.x * 64 + w * 4;   // first 64-block of this wave
    double m[4], t[32];
    bool gas[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int p = (b0 + u) * kBlk1 + lane;
        const bool in = p < nin;
        const int q = in ? p : 0;   // n > 0: particle 0 is there
        m[u] = in ? v.sm[q] : 0.0;
        const double x = v.sx[q], y = v.sy[q], z = v.sz[q];
        gas[u] = in && v.stype[q] == 2;
        t[8 * u] = m[u];
        t[8 * u + 1] = in ? x * m[u] : 0.0;
        t[8 * u + 2] = in ? y * m[u] : 0.0;
        t[8 * u + 3] = in ? z * m[u] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int p = (b0 + u) * kBlk1 + lane;
        t[8 * u + 4] = gas[u] ? m[u] : 0.0;
        t[8 * u + 5] = gas[u] ? v.svx[p] * m[u] : 0.0;
        t[8 * u + 6] = gas[u] ? v.svy[p] * m[u] : 0.0;
        t[8 * u + 7] = gas[u] ? v.svz[p] * m[u] : 0.0;
    }
    const double r = wave_sums32(t);
    if ((lane & 1) == 0) {
        const int j = lane >> 1;   // block b0 + (j >> 3), sum j & 7
        ((double *)(blk1 + b0))[j] = r;
        sb[j & 7][w * 4 + (j >> 3)] = r;
    }
    __syncthreads();
    if (w == 0) {
        double f[8];
#pragma unroll
        for (int j = 0; j < 8; j++) f[j] = sb[j][lane];
        const double q = wave_sums8(f);
        if ((lane & 7) == 0) ((double *)(blk2 + blockIdx.x))[lane >> 3] = q;
    }
}

// The greedy ascending cover of [s, e): head particles up to a 64-boundary,
// 64-blocks up to a 4096-boundary, 4096-blocks, 64-blocks, tail particles;
// then, for the parallel root, the particles [nin, n).
struct Cover {
    int s, h1, t2, t1, tail, p1, p2, p3, p4, nout, nin;
    int k1, k2, k3, k4, k5, total;
};

__device__ inline Cover make_cover(int s, int e, int nin, int nout) {
    Cover c;
    c.s = s;
    c.nin = nin;
    int a = (s + kBlk1 - 1) / kBlk1 * kBlk1;
    if (a > e) a = e;
    const int h0 = a - s;
    c.p1 = a;
    const int e1 = e / kBlk1 * kBlk1, e2 = e / kBlk2 * kBlk2;
    int b = (a + kBlk2 - 1) / kBlk2 * kBlk2;
    if (b > e1) b = e1 > a ? e1 : a;
    c.h1 = (b - a) / kBlk1;
    c.p2 = a + c.h1 * kBlk1;
    c.t2 = (c.p2 % kBlk2 == 0 && e2 > c.p2) ? (e2 - c.p2) / kBlk2 : 0;
    c.p3 = c.p2 + c.t2 * kBlk2;
    c.t1 = e1 > c.p3 ? (e1 - c.p3) / kBlk1 : 0;
    c.p4 = c.p3 + c.t1 * kBlk1;
    c.tail = e - c.p4;
    c.nout = nout;
    c.k1 = h0;
    c.k2 = c.k1 + c.h1;
    c.k3 = c.k2 + c.t2;
    c.k4 = c.k3 + c.t1;
    c.k5 = c.k4 + c.tail;
    c.total = c.k5 + nout;
    return c;
}

// The eight terms of piece k of a cover.  A particle and a block of sums are
// read through selected addresses, not on two branches, so a wave whose lanes
// hold both waits for memory once.
__device__ inline void load_piece(double (&f)[8], const Cover &c, int k, const PVals &v, const NodeSums *blk1,
                                  const NodeSums *blk2) {
    const bool part = k < c.k1 || k >= c.k4;
    const int p = k < c.k1 ? c.s + k : k < c.k5 ? c.p4 + (k - c.k4) : c.nin + (k - c.k5);
    const NodeSums *b = k < c.k2   ? blk1 + (c.p1 / kBlk1 + (k - c.k1))
                        : k < c.k3 ? blk2 + (c.p2 / kBlk2 + (k - c.k2))
                                   : blk1 + (c.p3 / kBlk1 + (k - c.k3));
    const int q = part ? p : 0;
    const double m = *(part ? v.sm + q : &b->m), g = *(part ? v.sm + q : &b->g);
    const double x = *(part ? v.sx + q : &b->sx), y = *(part ? v.sy + q : &b->sy), z = *(part ? v.sz + q : &b->sz);
    const double gx = *(part ? v.svx + q : &b->gx), gy = *(part ? v.svy + q : &b->gy),
                 gz = *(part ? v.svz + q : &b->gz);
    const bool gas = v.stype[q] == 2;
    f[0] = m;
    f[1] = part ? x * m : x;
    f[2] = part ? y * m : y;
    f[3] = part ? z * m : z;
    f[4] = part && !gas ? 0.0 : g;
    f[5] = part ? (gas ? gx * m : 0.0) : gx;
    f[6] = part ? (gas ? gy * m : 0.0) : gy;
    f[7] = part ? (gas ? gz * m : 0.0) : gz;
}

// Child-contiguous layout for the block walk (core::TreeNode): the root at 0,
// the children of node p at [1 + cstart[p], 1 + cstart[p] + nchild[p]) in
// octant order (rank, which in pre-order is the order of the children's first
// particles), cstart being the exclusive scan of nchild in pre-order.  A
// bucket (particles at one position) holds its member leaves, the next count
// nodes, as children.

// Every node at once: the sums over its key range (the parallel root also
// counts the particles outside its cube, Node.cpp:477-499), centre of mass,
// gas-weighted velocity, and the walk record at the node's layout place.
//
// PER nodes per workgroup, in XCD ranges (neighbours in pre-order share
// particles and blocks).  The particles of the workgroup's small nodes and
// leaves are staged in LDS once; the internal nodes are listed as small (up
// to kSumTiny particles, or more) and wide, so that the lanes of a wave loop
// over nodes of like size and the four waves share the wide ones; the sums
// pass to the nodes' own threads through LDS.  At 1,000,000 particles this is
// bound by memory (the node arrays and records, 150 to 210 bytes a node): sums and
// moments as two kernels, every node's lane looping over its own particles,
// took 65 + 110 us (17 + 5 us at 10,000), this one 91.
// A small tree takes 64 nodes per workgroup, whose wide nodes four waves then
// share: 14,800 nodes 9.2 us against 10.9 with 256, 48,000 11.1 against 12.0;
// 148,000 21.0 against 18.8, 1.48 M 119 against 92.
//
// Zero masses (zm, set when any particle has m == 0): the serial insert's
// running centre of mass (Node.cpp:692-697) divides by the node's mass after
// each particle; when the first particle to reach a node (the lowest caller
// index in it, since particles are inserted in array order) has m == 0, that
// is 0/0 and the node's centre stays NaN for good.  Such a node is never
// accepted (radius / NaN < theta is false), so the walk opens it.
constexpr int kSumTiny = 8;
constexpr int kMomentsSpread = 65536;   // up to this many nodes, 64 per workgroup

template <int PER>
__global__ __launch_bounds__(256) void k_node_moments(int nn, int nin, int n, int proot, int64_t thr, int zm,
                                                      const uint32_t *rid, DevState *ds,
                                                      const int32_t *first, const int32_t *count,
                                                      const int32_t *parent, const int32_t *pidx,
                                                      const int8_t *level, const NodeSums *blk1,
                                                      const NodeSums *blk2,
                                                      const double *gas_table, int gas_equal, int64_t ngas, PVals v,
                                                      const int32_t *nchild, const int32_t *rank,
                                                      const int32_t *cstart, double *gas_mass,
                                                      core::TreeNode *tree, core::SphNode *tsph,
                                                      int32_t *group_first, uint8_t *group_fired) {
    constexpr int kStage = PER + kSumSmall;   // particles staged
    __shared__ double st_m[kStage], st_x[kStage], st_y[kStage], st_z[kStage];
    __shared__ double st_vx[kStage], st_vy[kStage], st_vz[kStage];
    __shared__ uint8_t st_g[kStage];
    __shared__ double sum[8][PER];
    __shared__ int l_first[PER], l_count[PER];
    __shared__ uint8_t list[3][PER];   // tiny, small and wide nodes of this workgroup
    __shared__ int part[3][4];
    const int nd0 = xcd_block(blockIdx.x, gridDim.x) * PER;
    const int last = nd0 + PER - 1 < nn ? nd0 + PER - 1 : nn - 1;
    const int lane = lane_id(), wv = threadIdx.x >> 6;
    // PER < 256: the threads past PER own no node, and help with the sums
    const int nd = (int)threadIdx.x < PER ? nd0 + (int)threadIdx.x : nn;
    // every particle between the first particles of two nodes has its leaf
    // between them in pre-order, so the span is at most PER - 1 + kSumSmall
    const int P0 = first[nd0];
    int P1 = first[last] + kSumSmall;
    P1 = P1 < nin ? P1 : nin;
    int s = 0, cn = 0, p = -1;
    if (nd < nn) {
        s = first[nd];
        cn = count[nd];
        p = pidx[nd];
    }
    for (int k = threadIdx.x; k < P1 - P0; k += 256) {
        const int q = P0 + k;
        const bool g = v.stype[q] == 2;
        st_m[k] = v.sm[q]; st_x[k] = v.sx[q]; st_y[k] = v.sy[q]; st_z[k] = v.sz[q];
        st_g[k] = g ? 1 : 0;
        if (g) { st_vx[k] = v.svx[q]; st_vy[k] = v.svy[q]; st_vz[k] = v.svz[q]; }
    }
    const bool inner = nd < nn && p < 0;
    const bool wide = inner && ((nd == 0 && proot) || cn > kSumSmall);
    const bool tiny = inner && !wide && cn <= kSumTiny;
    const unsigned long long bal[3] = {__ballot(tiny), __ballot(inner && !wide && !tiny), __ballot(wide)};
    if (lane < 3) part[lane][wv] = __popcll(lane == 0 ? bal[0] : lane == 1 ? bal[1] : bal[2]);
    if ((int)threadIdx.x < PER) {
        l_first[threadIdx.x] = s;
        l_count[threadIdx.x] = cn;
    }
    __syncthreads();
    int len[3];
#pragma unroll
    for (int u = 0; u < 3; u++) {
        int at = 0;
        len[u] = 0;
        for (int k = 0; k < 4; k++) {
            const int h = part[u][k];
            at += k < wv ? h : 0;
            len[u] += h;
        }
        if (bal[u] >> lane & 1) list[u][at + __popcll(bal[u] & lanes_below())] = (uint8_t)threadIdx.x;
    }
    __syncthreads();
    // tiny and small nodes a lane each, in rows of 64
    const int rows0 = (len[0] + 63) / 64, rows = rows0 + (len[1] + 63) / 64;
    for (int r = wv; r < rows; r += 4) {
        const int u = r < rows0 ? 0 : 1;
        const int at = (r - (u ? rows0 : 0)) * 64 + lane;
        if (at < len[u]) {
            const int t = list[u][at];
            const int k0 = l_first[t] - P0, k1 = k0 + l_count[t];
            NodeSums a{0, 0, 0, 0, 0, 0, 0, 0};
            for (int k = k0; k < k1; k++) {
                const double m = st_m[k];
                a.m += m;
                a.sx += st_x[k] * m;
                a.sy += st_y[k] * m;
                a.sz += st_z[k] * m;
                if (st_g[k]) {
                    a.g += m;
                    a.gx += st_vx[k] * m;
                    a.gy += st_vy[k] * m;
                    a.gz += st_vz[k] * m;
                }
            }
            sum[0][t] = a.m; sum[1][t] = a.sx; sum[2][t] = a.sy; sum[3][t] = a.sz;
            sum[4][t] = a.g; sum[5][t] = a.gx; sum[6][t] = a.gy; sum[7][t] = a.gz;
        }
    }
    // wide nodes a wave each, the waves without rows first
    for (int j = 3 - wv; j < len[2]; j += 4) {
        const int t = list[2][j];
        const int ws = l_first[t];
        const bool root = nd0 + t == 0 && proot;
        const Cover cv = make_cover(ws, ws + l_count[t], nin, root ? n - nin : 0);
        double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        // two pieces in flight, added in order
        for (int k = lane; k < cv.total; k += 128) {
            const bool two = k + 64 < cv.total;
            double f[8], h[8];
            load_piece(f, cv, k, v, blk1, blk2);
            load_piece(h, cv, two ? k + 64 : k, v, blk1, blk2);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                a[i] += f[i];
                a[i] = two ? a[i] + h[i] : a[i];
            }
        }
        const double r = wave_sums8(a);
        if ((lane & 7) == 0) sum[lane >> 3][t] = r;
    }
    __syncthreads();
    if (nd >= nn) return;
    // cleared group state for the density phase (Node.cpp:722-796)
    group_first[nd] = kGroupNone;
    group_fired[nd] = 0;
    if (!tsph && nd == 0) ds->final_count = 0;   // no gas: no group in effect
    int par = parent[nd];
    double M, g, cx, cy, cz, mvx = 0.0, mvy = 0.0, mvz = 0.0;
    const core::Pos pos{v.sx, v.sy, v.sz};
    // buckets exist only where k_lcp met adjacent particles at one position
    const bool buckets = ds->any_bucket != 0;
    if (p >= 0) {
        const int k = p - P0;
        M = st_m[k];
        g = st_g[k] ? M : 0.0;
        bool vec = par < 0 ? (n == 1) : core::parallel_node(count, parent, par, n, thr);
        if (par >= 0 && !vec && buckets) {
            // members of a bucket sit exactly at their position
            const int ps = (par == 0 && proot) ? 0 : first[par];
            const int pe = (par == 0 && proot) ? n : first[par] + count[par];
            vec = core::is_bucket(pos, ps, pe);
        }
        cx = core::leaf_com(st_x[k], M, vec);
        cy = core::leaf_com(st_y[k], M, vec);
        cz = core::leaf_com(st_z[k], M, vec);
    } else {
        int e = s + cn;
        if (nd == 0 && proot) { s = 0; e = n; }
        double S[8];
#pragma unroll
        for (int j = 0; j < 8; j++) S[j] = sum[j][threadIdx.x];
        M = S[0];
        // equal gas masses: the reference's running sum, bit for bit (its
        // group selection compares gas masses and can sit on exact ties).
        // The node's gas count is its exactly rounded gas mass over the
        // common mass, rounded to the nearest integer (exact below 2^51).
        g = S[4];
        if (gas_equal && g > 0.0) {
            double q = rint(g / gas_table[1]);
            int64_t k = q < 0.0 ? 0 : (q > (double)ngas ? ngas : (int64_t)q);
            g = gas_table[k];
        }
        if (M > 0) { cx = S[1] / M; cy = S[2] / M; cz = S[3] / M; }
        else { cx = cy = cz = 0.0; }
        if (zm && !(nd == 0 && proot) && !core::parallel_node(count, parent, nd, n, thr)) {
            uint32_t first_any = 0xffffffffu, first_pos = 0xffffffffu;
            for (int j = s; j < s + cn; j++) {
                const uint32_t q = rid[j];
                first_any = q < first_any ? q : first_any;
                if (v.sm[j] != 0.0) first_pos = q < first_pos ? q : first_pos;
            }
            if (first_any < first_pos) cx = cy = cz = __builtin_nan("");
        }
        if (g > 0) { mvx = S[5] / g; mvy = S[6] / g; mvz = S[7] / g; }
        if (buckets && core::is_bucket(pos, s, e)) { cx = v.sx[s]; cy = v.sy[s]; cz = v.sz[s]; }
    }
    if (tsph) gas_mass[nd] = g;   // (pre-order: the density phase climbs it)
    const int place = core::node_place(nd, par, cstart, rank);
    const int kc = nchild[nd];
    core::TreeNode t;
    t.cx = cx; t.cy = cy; t.cz = cz; t.mass = M; t.gas = g;
    t.first_child = kc > 0 ? 1 + cstart[nd] : -1;
    t.nchild = kc;
    t.pidx = p;
    t.pre = nd;
    t.level = level[nd];
    t.flags = 0;
    t.pad0 = 0;
    t.pad1 = 0;
    tree[place] = t;
    if (tsph && g > 0.0) {   // only gas nodes are ever SPH candidates
        core::SphNode w;
        w.cx = cx; w.cy = cy; w.cz = cz; w.gas = g;
        if (p >= 0) { w.vx = st_vx[p - P0]; w.vy = st_vy[p - P0]; w.vz = st_vz[p - P0]; }
        else { w.vx = mvx; w.vy = mvy; w.vz = mvz; }
        w.pidx = p;
        w.pad = 0;
        tsph[place] = w;
    }
}

// Exclusive scan of an int array of host-known length (tiles of 1024).
__global__ __launch_bounds__(256) void k_iscan_tiles(int n, const int32_t *in, int32_t *bsum) {
    __shared__ int scr[4];
    int b0 = blockIdx.x * 1024 + threadIdx.x * 4;
    int s = 0;
    for (int k = 0; k < 4; k++) s += (b0 + k < n) ? in[b0 + k] : 0;
    int tot;
    block256_excl_scan(s, scr, &tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// In a build's scan of the children (ds given) the first workgroup also folds
// the leaves' partials.
__global__ __launch_bounds__(256) void k_iscan_apply(int n, const int32_t *in, const int32_t *bsum, int32_t *out,
                                                     int nleaf_tiles, const int32_t *leaf_part, DevState *ds) {
    __shared__ int scr[4];
    if (ds && blockIdx.x == 0) leaf_fold(nleaf_tiles, leaf_part, ds);
    int b0 = blockIdx.x * 1024 + threadIdx.x * 4;
    int v[4];
    int s = 0;
    for (int k = 0; k < 4; k++) { v[k] = (b0 + k < n) ? in[b0 + k] : 0; s += v[k]; }
    const int pre = tile_offset(bsum, (int)gridDim.x, (int)blockIdx.x, scr, nullptr);
    int ex = block256_excl_scan(s, scr, nullptr) + pre;
    for (int k = 0; k < 4; k++) {
        if (b0 + k < n) out[b0 + k] = ex;
        ex += v[k];
    }
}

// ------------------------------------------------------------ deep refinement
// Distinct particles that agree on every key word so far, and tie runs too
// long for k_tie_rank, are refined word by word: the particles tied on words
// 0..w-1 get word w and each tie run is sorted by (word w, caller index)
// with a general segmented LSD radix sort over just those particles
// (compacted; run start, word and caller index as three stable sorts).
// Runs sit at contiguous positions, so the k-th particle of the sorted
// compact list takes the k-th compact position.  All of it works on the
// order before the state permutation (ord = the sort permutation).
__device__ inline bool words_equal(const core::KeyWords &kw, int a, int b, int w) {
    for (int j = 0; j < w; j++)
        if (kw.w[j][a] != kw.w[j][b]) return false;
    return true;
}

__device__ inline int tie_first(const core::KeyWords &kw, int w, int i) {
    int hi = i, lo = -1;
    for (int step = 1;; step <<= 1) {
        const int probe = i - step;
        if (probe < 0) break;
        if (!words_equal(kw, probe, i, w)) { lo = probe; break; }
        hi = probe;
        if (step > (1 << 29)) break;
    }
    while (hi - lo > 1) {
        const int mid = lo + ((hi - lo) >> 1);
        if (words_equal(kw, mid, i, w)) hi = mid; else lo = mid;
    }
    return hi;
}

// flag[i] = 1 if particle i shares words 0..w-1 with a neighbour
__global__ __launch_bounds__(256) void k_deep_flag(const DevState *ds, core::KeyWords kw, int w, int32_t *flag) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int nin = ds->nin;
    if (i >= nin) return;
    const bool t = (i > 0 && words_equal(kw, i - 1, i, w)) || (i + 1 < nin && words_equal(kw, i, i + 1, w));
    flag[i] = t ? 1 : 0;
}

__global__ __launch_bounds__(256) void k_deep_compact(const DevState *ds, const int32_t *flag, const int32_t *offs,
                                                      uint32_t *spos, int32_t *m_out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int nin = ds->nin;
    if (i >= nin) return;
    if (flag[i]) spos[offs[i]] = (uint32_t)i;
    if (i == nin - 1) *m_out = offs[i] + flag[i];
}

// Word w of every flagged particle (w >= 2; word 1 exists already), its
// run start, and the first sort key (caller index).
__global__ __launch_bounds__(256) void k_deep_word(int m, const uint32_t *spos, const uint32_t *ord,
                                                   const double *x, const double *y, const double *z,
                                                   const uint32_t *rid, const DevState *ds, core::KeyWords kw,
                                                   int w, uint64_t *word_w, uint8_t *gapl, uint32_t *srun,
                                                   uint64_t *sk, uint32_t *sv) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= m) return;
    const int i = (int)spos[k];
    const uint32_t q = ord[i];
    if (w >= 2) {
        const double R = __longlong_as_double((long long)ds->Rbits);
        int g = 0;
        word_w[i] = core::octant_word(x[q], y[q], z[q], R, w, &g);
        if (gapl[q] == 0 && g > 0) gapl[q] = (uint8_t)(g > 254 ? 254 : g);
    }
    srun[k] = (uint32_t)tie_first(kw, w, i);
    sk[k] = (uint64_t)rid[q];
    sv[k] = (uint32_t)k;
}

// sk[j] = word w of the compact element sv[j] (second sort key)
__global__ __launch_bounds__(256) void k_deep_key_word(int m, const uint32_t *sv, const uint32_t *spos,
                                                       const uint64_t *word_w, uint64_t *sk) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < m) sk[j] = word_w[spos[sv[j]]];
}

// sk[j] = run start of the compact element sv[j] (third sort key)
__global__ __launch_bounds__(256) void k_deep_key_run(int m, const uint32_t *sv, const uint32_t *srun, uint64_t *sk) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < m) sk[j] = (uint64_t)srun[sv[j]];
}

// The j-th sorted element moves to the j-th compact position.
__global__ __launch_bounds__(256) void k_deep_scatter(int m, const uint32_t *spos, const uint32_t *sv,
                                                      const uint32_t *ord, const uint64_t *word_w, uint32_t *ord_tmp,
                                                      uint64_t *word_tmp) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= m) return;
    const uint32_t dst = spos[j], src = spos[sv[j]];
    ord_tmp[dst] = ord[src];
    word_tmp[dst] = word_w[src];
}

__global__ __launch_bounds__(256) void k_deep_back(int m, const uint32_t *spos, const uint32_t *ord_tmp,
                                                   const uint64_t *word_tmp, uint32_t *ord, uint64_t *word_w) {
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= m) return;
    const uint32_t p = spos[j];
    ord[p] = ord_tmp[p];
    word_w[p] = word_tmp[p];
}

__global__ void k_reset_tie_flags(DevState *ds) {
    ds->tie_big = 0;
    ds->tie_deep = 0;
}

// Internal children of every node, for k_branch_depth (zeroed, then counted).
__global__ __launch_bounds__(256) void k_zero_inner(int nn, int32_t *ichild, DevState *ds) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < nn) ichild[p] = 0;
    if (p == 0) ds->walk_depth = 0;
}

__global__ __launch_bounds__(256) void k_count_inner(int nn, const int32_t *pidx, const int32_t *parent,
                                                     int32_t *ichild) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < nn && pidx[p] < 0 && parent[p] >= 0) atomicAdd(&ichild[parent[p]], 1);
}

// Stack growth bound of the block walk in a deep tree.  Taking one block of
// siblings off the stack pushes one block per sibling opened, and only
// internal nodes are opened, so the stack grows by at most (internal
// children - 1) at a node; along any root-to-leaf path the sum of those is
// the most the stack can grow below a point (the walk adds 8 of slack).
// Chains of single-internal-child cells (a galaxy far down a root cube
// stretched by escaped particles, with a stray particle beside each level)
// add nothing.
__global__ __launch_bounds__(256) void k_branch_depth(int nin, const int32_t *base, const int32_t *c,
                                                      const int32_t *parent, const int32_t *ichild, DevState *ds) {
    __shared__ int wmax[4];
    const int i = blockIdx.x * 256 + threadIdx.x;
    int d = 0;
    if (i < nin) {
        const int leaf = i + base[i] + c[i];
        for (int a = parent[leaf]; a >= 0; a = parent[a]) d += ichild[a] > 1 ? ichild[a] - 1 : 0;
        d += 8;
    }
    for (int o = 32; o >= 1; o >>= 1) {
        const int t = __shfl_xor(d, o, 64);
        d = t > d ? t : d;
    }
    if (lane_id() == 0) wmax[threadIdx.x >> 6] = d;
    __syncthreads();
    if (threadIdx.x == 0) {
        int b = wmax[0];
        for (int k = 1; k < 4; k++) b = wmax[k] > b ? wmax[k] : b;
        atomicMax(&ds->walk_depth, b);
    }
}

}  // namespace

void alloc_nodes(Ctx &c, int64_t cap) {
    reset_graphs(c);   // the node capacity is an argument of the captured segments
    if (c.node_slab) {
        (void)hipFree(c.node_slab);
        c.node_slab = nullptr;
    }
    c.node_cap = cap;
    const size_t n = (size_t)cap;
    // block sums for every particle slot (launch_tile_sums covers all c.n <= c.cap)
    const size_t pcap = (size_t)c.cap > n ? (size_t)c.cap : n;
    auto plan = [&](Carve &cv) {
        cv(&c.n_first, n * 4); cv(&c.n_count, n * 4);
        cv(&c.n_parent, n * 4);
        cv(&c.n_pidx, n * 4); cv(&c.n_level, n);
        cv(&c.n_gas, n * 8); cv(&c.g_rho, n * 8);
        cv(&c.g_first, n * 4); cv(&c.g_list, (n + 256) * 4);
        cv(&c.g_fired, n); cv(&c.g_final, n * 4);
        cv(&c.tnode, n * sizeof(core::TreeNode));
        cv(&c.tsph, n * sizeof(core::SphNode));
        cv(&c.n_nchild, n * 4); cv(&c.n_rank, n * 4); cv(&c.n_cstart, n * 4);
        cv(&c.nsum_tile, (pcap / kBlk2 + 1) * (kBlk2 / kBlk1 + 1) * sizeof(NodeSums));
        cv(&c.n_bsum, (n / 1024 + 2) * 4);
    };
    Carve size;
    plan(size);
    AG2_HIP(hipMalloc(&c.node_slab, size.off));
    Carve at;
    at.base = (char *)c.node_slab;
    plan(at);
}

void state_fields(Ctx &c, double **f[kStateD]) {
    double **l[kStateD] = {&c.x, &c.y, &c.z, &c.vx, &c.vy, &c.vz, &c.m, &c.U, &c.mu, &c.ax,
                           &c.ay, &c.az, &c.h, &c.rho, &c.P, &c.T, &c.dUdt, &c.ts, &c.next};
    static_assert(kAccField == 9 && kHField == 12, "field order: accelerations after nine fields, then h");
    for (int j = 0; j < kStateD; j++) f[j] = l[j];
}

// The permutation into key order writes the alternate buffers; swap_state
// then makes them current on the host side (also when the launch came from
// a replayed graph).
static void launch_permute(Ctx &c, int n) {
    double **f[kStateD];
    state_fields(c, f);
    StateSet in, out;
    for (int j = 0; j < kStateD; j++) { in.d[j] = *f[j]; out.d[j] = c.alt[j]; }
    in.type = c.type; in.active = c.active; in.rid = c.rid;
    out.type = c.type_alt; out.active = c.active_alt; out.rid = c.rid_alt;
    // idx_alt: the sort permutation after the tie runs' order (k_tie_rank).
    // A captured segment keeps its arguments for every replay, so graph
    // launches always move the accelerations.
    const int skip_acc = c.acc_overwritten && !c.p.graph_launch ? 1 : 0;
    const int zero_gas_h = c.density_follows && !c.p.graph_launch ? 1 : 0;
    c.h_cleared = zero_gas_h != 0;
    const unsigned g = grid_for(n, 256);
    if (n <= kPermuteSplit)
        hipLaunchKernelGGL(k_permute<kPermuteParts>, dim3(g, kPermuteParts), dim3(256), 0, c.stream, n, c.idx_alt, in,
                           out, skip_acc, zero_gas_h);
    else
        hipLaunchKernelGGL(k_permute<1>, dim3(g), dim3(256), 0, c.stream, n, c.idx_alt, in, out, skip_acc, zero_gas_h);
}

static void swap_state(Ctx &c) {
    double **f[kStateD];
    state_fields(c, f);
    for (int j = 0; j < kStateD; j++) std::swap(*f[j], c.alt[j]);
    std::swap(c.type, c.type_alt);
    std::swap(c.active, c.active_alt);
    std::swap(c.rid, c.rid_alt);
    c.parity ^= 1;
}

void build_inverse(Ctx &c) {
    hipLaunchKernelGGL(k_inverse, dim3(grid_for(c.n, 256)), dim3(256), 0, c.stream, (int)c.n, c.rid, c.inv);
    AG2_HIP(hipGetLastError());
}

// LSD radix passes over (key, value) pairs, 8-bit digits from bit shift0:
// an even number of passes leaves the result in kin / vin.
static void radix_pairs(Ctx &c, int n, uint64_t *kin, uint64_t *kout, uint32_t *vin, uint32_t *vout, int shift0,
                        int passes) {
    const int nblk = (n + kSortTile - 1) / kSortTile;
    if (nblk < 1) return;
    const bool small = nblk <= kSortSmallTiles;
    for (int pass = 0; pass < passes; pass++) {
        const int shift = shift0 + pass * 8;
        hipLaunchKernelGGL(k_rs_hist, dim3(nblk), dim3(256), 0, c.stream, n, kin, shift, c.hist, nblk);
        if (small) {
            hipLaunchKernelGGL(k_rs_scatter<true>, dim3(nblk), dim3(256), 0, c.stream, n, kin, vin, kout, vout, shift,
                               c.hist, c.dtotal, nblk);
        } else {
            hipLaunchKernelGGL(k_rs_scan, dim3(256), dim3(256), 0, c.stream, nblk, c.hist, c.dtotal);
            hipLaunchKernelGGL(k_rs_scatter<false>, dim3(nblk), dim3(256), 0, c.stream, n, kin, vin, kout, vout, shift,
                               c.hist, c.dtotal, nblk);
        }
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
}

template <int TILE>
static void merge_sort(Ctx &c, int n) {
    hipLaunchKernelGGL(k_ms_tile<TILE>, dim3(grid_for(n, TILE)), dim3(kMsThreads), 0, c.stream, n, c.key, c.idx,
                       c.key_alt, c.idx_alt, c.sort_lo, (uint64_t *)nullptr, 0);
    if constexpr (TILE == kMsTiny0)
        hipLaunchKernelGGL(k_ms_merge_lds, dim3(grid_for(n, kMsThreads / kMsLanes)), dim3(kMsThreads), 0, c.stream, n,
                           c.key_alt, c.idx_alt, c.key, c.idx, c.sort_lo);
    else
        hipLaunchKernelGGL(k_ms_merge<TILE>, dim3(grid_for(n, kMsPer)), dim3(256), 0, c.stream, n, c.key_alt, c.idx_alt,
                           c.key, c.idx, c.sort_lo);
}

template <int TILE, int ITEMS>
static void sample_sort(Ctx &c, int n, int step) {
    // samples and splitters in key2, which is written after the sort
    const int tiles = grid_for(n, TILE), S = TILE / step;
    Splitter *split = (Splitter *)(c.key2 + (size_t)tiles * S);
    hipLaunchKernelGGL(k_ms_tile<TILE>, dim3(tiles), dim3(kMsThreads), 0, c.stream, n, c.key, c.idx, c.key_alt,
                       c.idx_alt, c.sort_lo, c.key2, step);
    hipLaunchKernelGGL(k_bs_split<TILE>, dim3(tiles), dim3(kMsThreads), 0, c.stream, n, step, c.key2, split);
    hipLaunchKernelGGL((k_bs_bucket<TILE, ITEMS>), dim3(tiles * S / kBsPer), dim3(kMsThreads), 0, c.stream, n, step,
                       c.key_alt, c.idx_alt, c.key, c.idx, c.sort_lo, split);
}

static void radix_sort(Ctx &c, int n) {
    int nblk = (n + kSortTile - 1) / kSortTile;
    uint64_t *kin = c.key, *kout = c.key_alt;
    uint32_t *vin = c.idx, *vout = c.idx_alt;
    if (n <= kMsMax) {
        if (n <= kMsTiny) merge_sort<kMsTiny0>(c, n);
        else if (n <= kMsSmall) merge_sort<kMsTile0>(c, n);
        else merge_sort<kMsTile1>(c, n);
        return;
    }
    if (n <= kBsMax) {
        const int step = bs_step(n);
        if (step == 16) sample_sort<kMsTile0, 2>(c, n, step);
        else if (step == 32) sample_sort<kMsTile0, 4>(c, n, step);
        else sample_sort<kMsTile1, 8>(c, n, step);
        return;
    }
    // bytes sort_lo .. 7 (an even number of passes)
    for (int pass = c.sort_lo; pass < 8; pass++) {
        int shift = pass * 8;
        hipLaunchKernelGGL(k_rs_hist, dim3(nblk), dim3(256), 0, c.stream, n, kin, shift, c.hist, nblk);
        hipLaunchKernelGGL(k_rs_scan, dim3(256), dim3(256), 0, c.stream, nblk, c.hist, c.dtotal);
        hipLaunchKernelGGL(k_rs_scatter<false>, dim3(nblk), dim3(256), 0, c.stream, n, kin, vin, kout, vout, shift,
                           c.hist, c.dtotal, nblk);
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    // an even number of passes: the result is back in c.key / c.idx
    static_assert(kSortLoMax % 2 == 0, "the sort must end in its input buffers");
}

// First half of the build in three launch segments.  Their kernel
// arguments depend only on the particle count, the node capacity, the
// parameters and the state parity, so with ag2_params.graph_launch each
// segment is captured once per parity as a HIP graph and replayed; by
// default every kernel is launched on its own.  No segment holds a memset.
static void seg_keys(Ctx &c) {
    int n = (int)c.n;
    hipStream_t st = c.stream;
    int g = grid_for(n, 256);
    int twb = g < kTwBlocks ? (g > 0 ? g : 1) : kTwBlocks;
    // partials: the sums at [0, 2 twb), the maxima after them
    unsigned long long *rmax = (unsigned long long *)(c.partials + 2 * kTwBlocks);
    if (!c.tw_partials) hipLaunchKernelGGL(k_tw_partial, dim3(twb), dim3(256), 0, st, n, c.x, c.y, c.z, c.partials);
    c.tw_partials = false;
    hipLaunchKernelGGL(k_tw_max, dim3(twb), dim3(256), 0, st, n, c.x, c.y, c.z, twb, c.partials, c.ds, rmax);
    hipLaunchKernelGGL(k_keygen, dim3(g), dim3(256), 0, st, n, c.x, c.y, c.z, twb, rmax, c.ds, c.key, c.idx,
                       c.gapl);
}

static void seg_sort(Ctx &c) { radix_sort(c, (int)c.n); }

static void seg_order(Ctx &c) {
    int n = (int)c.n;
    hipStream_t st = c.stream;
    int g = grid_for(n, 256);
    const int shift = 8 * c.sort_lo;
    hipLaunchKernelGGL(k_tie_key2, dim3(g), dim3(256), 0, st, n, c.key, c.idx, c.x, c.y, c.z, c.ds, c.key2, c.gapl,
                       shift);
    // word 1 in run order -> key_alt, the permutation -> idx_alt
    hipLaunchKernelGGL(k_tie_rank, dim3(g), dim3(256), 0, st, n, c.key, c.key2, c.idx, c.rid, c.ds, c.w0, c.key_alt,
                       c.idx_alt, shift);
    launch_permute(c, n);
    int proot = (c.n >= 2 && c.n >= c.p.split_threshold) ? 1 : 0;
    // from here on the state is the permuted one (alternate buffers)
    core::KeyWords kw{{c.w0, c.key_alt, nullptr, nullptr, nullptr, nullptr}};
    core::Pos pos{c.alt[0], c.alt[1], c.alt[2]};
    int nb = (n + 1023) / 1024;
    if (nb < 1) nb = 1;
    hipLaunchKernelGGL(k_lcp, dim3(nb), dim3(kLevTile), 0, st, n, kw, 2, pos, c.ds, proot, c.lcp, c.lmin, c.cnt,
                       c.bsum);
    hipLaunchKernelGGL(k_scan_apply, dim3(nb), dim3(256), 0, st, c.cnt, c.bsum, c.ds, proot, c.node_cap, c.base);
    AG2_HIP(hipMemcpyAsync(c.hs_pinned, c.ds, sizeof(DevState), hipMemcpyDeviceToHost, st));
}

void reset_graphs(Ctx &c) {
    for (auto &row : c.seg_exec)
        for (auto &e : row)
            if (e) {
                (void)hipGraphExecDestroy(e);
                e = nullptr;
            }
}

static void run_segment(Ctx &c, int s, void (*fn)(Ctx &)) {
    if (!c.p.graph_launch) {
        fn(c);
        AG2_HIP(hipGetLastError());
        return;
    }
    hipGraphExec_t &ex = c.seg_exec[s][s == 1 ? 0 : c.parity];
    if (!ex) {
        hipGraph_t gr = nullptr;
        AG2_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
        try {
            fn(c);
        } catch (...) {
            // leave the stream out of capture mode before the error goes up
            hipGraph_t dead = nullptr;
            (void)hipStreamEndCapture(c.stream, &dead);
            if (dead) (void)hipGraphDestroy(dead);
            throw;
        }
        hipError_t le = hipGetLastError();
        hipError_t ce = hipStreamEndCapture(c.stream, &gr);
        AG2_HIP(le);
        AG2_HIP(ce);
        hipError_t ie = hipGraphInstantiate(&ex, gr, nullptr, nullptr, 0);
        (void)hipGraphDestroy(gr);
        if (ie != hipSuccess) ex = nullptr;
        AG2_HIP(ie);
    }
    AG2_HIP(hipGraphLaunch(ex, c.stream));
}

// First half of the build, up to the node count, and the particle prefix
// sums: everything here is asynchronous; the state it leaves in c.ds (nin,
// n_int, n_nodes, err) is copied to c.hs_pinned, and c.ev_counts completes
// when it is there -- build_tree_b must not start before.
void build_keys(Ctx &c) {
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[0], c.stream));
    run_segment(c, 0, seg_keys);
}

void build_tree_a(Ctx &c) {
    build_keys(c);
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[1], c.stream));
    run_segment(c, 1, seg_sort);
    build_order(c);
}

size_t sort_job_bytes() { return sizeof(SortJob); }

template <int TILE>
static void merge_batch(int tiles, const SortJob *dj, int nc, int lo, hipStream_t st) {
    hipLaunchKernelGGL(k_msb_tile<TILE>, dim3(tiles), dim3(kMsThreads), 0, st, dj, nc, lo, 0);
    hipLaunchKernelGGL(k_msb_merge<TILE>, dim3((unsigned)(tiles * (TILE / kMsPer))), dim3(256), 0, st, dj, nc, lo);
}

void sort_batch(Ctx *const *cs, int nc, hipStream_t st, void *scratch_dev, void *scratch_host) {
    if (nc <= 0) return;
    SortJob *hj = (SortJob *)scratch_host;
    // the bytes every job sorts (an even number of passes ends in key / idx),
    // and by which sort: each job's order is that of its own sort either way
    int lo = kSortLoMax;
    int64_t most = 0;
    for (int k = 0; k < nc; k++) {
        lo = cs[k]->sort_lo < lo ? cs[k]->sort_lo : lo;
        most = cs[k]->n > most ? cs[k]->n : most;
    }
    const int tile = most > kBsBatchMax                         ? kSortTile
                     : most <= kMsTiny                     ? kMsTiny0
                     : most > kMsMax || most <= kMsSmall ? kMsTile0
                                                           : kMsTile1;
    int total = 0;
    for (int k = 0; k < nc; k++) {
        Ctx &c = *cs[k];
        const int n = (int)c.n;
        const int nblk = (n + tile - 1) / tile;
        hj[k] = SortJob{n, nblk, total, 0, c.key, c.key_alt, c.idx, c.idx_alt, c.hist, c.dtotal, c.key2};
        total += nblk;
    }
    if (total < 1) return;
    SortJob *dj = (SortJob *)scratch_dev;
    AG2_HIP(hipMemcpyAsync(dj, hj, sizeof(SortJob) * (size_t)nc, hipMemcpyHostToDevice, st));
    if (most <= kMsMax) {
        if (tile == kMsTiny0) merge_batch<kMsTiny0>(total, dj, nc, lo, st);
        else if (tile == kMsTile0) merge_batch<kMsTile0>(total, dj, nc, lo, st);
        else merge_batch<kMsTile1>(total, dj, nc, lo, st);
        AG2_HIP(hipGetLastError());
        return;
    }
    if (most <= kBsBatchMax) {
        const dim3 g(total), b(kMsThreads);
        hipLaunchKernelGGL(k_msb_tile<kMsTile0>, g, b, 0, st, dj, nc, lo, kMsTile0 / kBsPer);
        hipLaunchKernelGGL(k_bsb_split<kMsTile0>, g, b, 0, st, dj, nc);
        hipLaunchKernelGGL((k_bsb_bucket<kMsTile0, 4>), g, b, 0, st, dj, nc, lo);
        AG2_HIP(hipGetLastError());
        return;
    }
    for (int pass = lo; pass < 8; pass++) {
        hipLaunchKernelGGL(k_rsb_hist, dim3(total), dim3(256), 0, st, dj, nc, pass);
        hipLaunchKernelGGL(k_rsb_scan, dim3(256 * nc), dim3(256), 0, st, dj);
        hipLaunchKernelGGL(k_rsb_scatter, dim3(total), dim3(256), 0, st, dj, nc, pass);
    }
    // every job's result is back in its key / idx
    AG2_HIP(hipGetLastError());
}

// The block sums of the node-sum cover (k_tile_sums), laid out for all n
// particles: 64-blocks, then 4096-blocks.
static void tile_sum_buffers(const Ctx &c, NodeSums **blk1, NodeSums **blk2) {
    const int64_t ntile = (c.n + kBlk2 - 1) / kBlk2;
    *blk1 = c.nsum_tile;
    *blk2 = c.nsum_tile + (size_t)ntile * (kBlk2 / kBlk1);
}

static void launch_tile_sums(Ctx &c) {
    const int ntile = (int)((c.n + kBlk2 - 1) / kBlk2);
    if (ntile < 1) return;
    NodeSums *blk1, *blk2;
    tile_sum_buffers(c, &blk1, &blk2);
    PVals pv{c.x, c.y, c.z, c.m, c.vx, c.vy, c.vz, c.type};
    hipLaunchKernelGGL(k_tile_sums, dim3(ntile), dim3(1024), 0, c.stream, c.ds, pv, blk1, blk2);
}

static NodeArrays node_arrays(const Ctx &c) {
    return NodeArrays{c.n_first, c.n_count, c.n_parent, c.n_pidx, c.n_nchild, c.n_rank, c.n_level};
}

// n_cstart lists the internal nodes' particles until the child-place scan
// overwrites it.
static void launch_leaves(Ctx &c) {
    const int nb = ((int)c.n + kLevTile - 1) / kLevTile;
    if (nb < 1) return;
    hipLaunchKernelGGL(k_make_leaf, dim3(nb), dim3(kLevTile), 0, c.stream, c.ds, c.lcp, c.base, c.cnt, node_arrays(c),
                       c.idx_alt, c.gapl, c.n_cstart, c.n_bsum, c.leaf_part);
}

// Up to 65536 internal nodes (1024 workgroups of 64, four a CU) fewer nodes
// per workgroup spread the listed nodes over more waves: 10,000 particles 9.5
// us against 11.0 with 256 nodes, 100,000 12.7 against 13.5; 1,000,000 35
// against 30.
constexpr int kInternalSpread = 65536;

static void launch_internal(Ctx &c, const NodeArrays &o) {
    if (c.n_int <= kInternalSpread)
        hipLaunchKernelGGL(k_make_internal<64>, dim3(grid_for(c.n_int, 64)), dim3(256), 0, c.stream, c.nin, c.n_int,
                           c.lcp, c.lmin, c.base, c.n_cstart, o, c.n_bsum);
    else
        hipLaunchKernelGGL(k_make_internal<256>, dim3(grid_for(c.n_int, 256)), dim3(256), 0, c.stream, c.nin,
                           c.n_int, c.lcp, c.lmin, c.base, c.n_cstart, o, c.n_bsum);
}

void build_order(Ctx &c) {
    hipStream_t st = c.stream;
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[2], st));
    // poisoned until this build's counts overwrite it (checked in build_tree_b)
    c.hs_pinned->n_nodes = -1;
    run_segment(c, 2, seg_order);
    swap_state(c);
    AG2_HIP(hipEventRecord(c.ev_counts, st));
    // the leaves and the block sums need only the particles in key order:
    // they run while the host waits for the counts
    launch_leaves(c);
    launch_tile_sums(c);
    AG2_HIP(hipGetLastError());
}

core::KeyWords key_words(const Ctx &c) {
    core::KeyWords kw{{c.w0, c.key_alt, nullptr, nullptr, nullptr, nullptr}};
    for (int w = 2; w < c.kw_used; w++) kw.w[w] = c.kdeep[w - 2];
    return kw;
}

// Buffers of the deep refinement, allocated on its first use.
static void alloc_deep(Ctx &c) {
    if (c.sk) return;
    const size_t n = (size_t)c.cap;
    for (uint64_t *&p : c.kdeep) AG2_HIP(hipMalloc(&p, n * 8));
    AG2_HIP(hipMalloc(&c.sk, n * 8));
    AG2_HIP(hipMalloc(&c.sk_alt, n * 8));
    AG2_HIP(hipMalloc(&c.sv, n * 4));
    AG2_HIP(hipMalloc(&c.sv_alt, n * 4));
    AG2_HIP(hipMalloc(&c.spos, n * 4));
    AG2_HIP(hipMalloc(&c.srun, n * 4));
}


// The slow path of a build, taken only when the first half flagged a tie
// run longer than k_tie_rank's bound or distinct particles that agree on
// both key words (the reference splits such cells until they separate,
// Node.cpp:597-699).  The first half's permutation read the state without
// changing it, so the state goes back to its input buffers; the order is
// refined word by word (deep refinement kernels), and the state permuted,
// the topology counted and the prefix sums formed again.  Each word costs a
// few host reads; distinct particles still together after kDeepest levels
// fail the build.
static void refine_ties(Ctx &c) {
    hipStream_t st = c.stream;
    const int n = (int)c.n;
    const int nin = c.hs.nin;
    alloc_deep(c);
    swap_state(c);   // the state before this build's permutation
    const int g = grid_for(nin, 256);
    const int nb = (nin + 1023) / 1024;
    c.kw_used = 2;
    for (int w = c.hs.tie_big ? 1 : 2; w < core::kKeyWords; w++) {
        const core::KeyWords kw = key_words(c);   // words 0 .. w-1 are present
        hipLaunchKernelGGL(k_deep_flag, dim3(g), dim3(256), 0, st, c.ds, kw, w, c.cnt);
        hipLaunchKernelGGL(k_iscan_tiles, dim3(nb), dim3(256), 0, st, nin, c.cnt, c.bsum);
        hipLaunchKernelGGL(k_iscan_apply, dim3(nb), dim3(256), 0, st, nin, c.cnt, c.bsum, c.base, 0,
                           (const int32_t *)nullptr, (DevState *)nullptr);
        hipLaunchKernelGGL(k_deep_compact, dim3(g), dim3(256), 0, st, c.ds, c.cnt, c.base, c.spos, &c.ds->deep_m);
        AG2_HIP(hipMemcpyAsync(&c.hs_pinned->deep_m, &c.ds->deep_m, sizeof(int32_t), hipMemcpyDeviceToHost, st));
        AG2_HIP(hipStreamSynchronize(st));
        const int m = c.hs_pinned->deep_m;
        if (m <= 0) break;
        uint64_t *word_w = w == 1 ? c.key_alt : c.kdeep[w - 2];
        const unsigned gm = grid_for(m, 256);
        hipLaunchKernelGGL(k_deep_word, dim3(gm), dim3(256), 0, st, m, c.spos, c.idx_alt, c.x, c.y, c.z, c.rid, c.ds,
                           kw, w, word_w, c.gapl, c.srun, c.sk, c.sv);
        radix_pairs(c, m, c.sk, c.sk_alt, c.sv, c.sv_alt, 0, 4);   // caller index
        hipLaunchKernelGGL(k_deep_key_word, dim3(gm), dim3(256), 0, st, m, c.sv, c.spos, word_w, c.sk);
        radix_pairs(c, m, c.sk, c.sk_alt, c.sv, c.sv_alt, 0, 8);   // word w
        hipLaunchKernelGGL(k_deep_key_run, dim3(gm), dim3(256), 0, st, m, c.sv, c.srun, c.sk);
        radix_pairs(c, m, c.sk, c.sk_alt, c.sv, c.sv_alt, 0, 4);   // run start
        hipLaunchKernelGGL(k_deep_scatter, dim3(gm), dim3(256), 0, st, m, c.spos, c.sv, c.idx_alt, word_w, c.idx,
                           c.key2);
        hipLaunchKernelGGL(k_deep_back, dim3(gm), dim3(256), 0, st, m, c.spos, c.idx, c.key2, c.idx_alt, word_w);
        c.kw_used = w + 1 > c.kw_used ? w + 1 : c.kw_used;
    }
    hipLaunchKernelGGL(k_reset_tie_flags, dim3(1), dim3(1), 0, st, c.ds);
    launch_permute(c, n);
    const int proot = (c.n >= 2 && c.n >= c.p.split_threshold) ? 1 : 0;
    const core::Pos pos{c.alt[0], c.alt[1], c.alt[2]};
    const int nbn = (n + 1023) / 1024 < 1 ? 1 : (n + 1023) / 1024;
    hipLaunchKernelGGL(k_lcp, dim3(nbn), dim3(kLevTile), 0, st, n, key_words(c), c.kw_used, pos, c.ds,
                       proot, c.lcp, c.lmin, c.cnt, c.bsum);
    hipLaunchKernelGGL(k_scan_apply, dim3(nbn), dim3(256), 0, st, c.cnt, c.bsum, c.ds, proot, c.node_cap, c.base);
    swap_state(c);
    AG2_HIP(hipMemcpyAsync(c.hs_pinned, c.ds, sizeof(DevState), hipMemcpyDeviceToHost, st));
    AG2_HIP(hipStreamSynchronize(st));
    c.hs = *c.hs_pinned;
    if (c.hs.tie_deep)
        throw CapacityError("distinct particles share all 126 octant levels of the root cube (closer than 2^-126 "
                            "of its half-width); the reference would keep splitting them (Node.cpp:597-699)");
}

// Second half: nodes, moments and the walk layout, sized by the counts the
// first half left in c.hs_pinned (c.ev_counts has completed since; the
// prefix sums queued after it may still run).
void build_tree_b(Ctx &c) {
    int n = (int)c.n;
    hipStream_t st = c.stream;
    int proot = (c.n >= 2 && c.n >= c.p.split_threshold) ? 1 : 0;
    c.hs = *c.hs_pinned;
    if (c.hs.n_nodes < 0) throw HipError("the node counts of this build did not reach the host");
    if (c.hs.tie_big && c.sort_lo > 0) {
        // a run of particles sharing the sorted bits too long for the
        // ranking: the first half again, sorting every byte of word 0
        c.sort_lo = 0;
        build_tree_a(c);
        AG2_HIP(hipEventSynchronize(c.ev_counts));
        c.hs = *c.hs_pinned;
        if (c.hs.n_nodes < 0) throw HipError("the node counts of this build did not reach the host");
    } else if (!c.p.graph_launch) {
        // the next build leaves the low bytes out again unless its runs got long
        c.sort_lo = c.hs.max_prefix_run > kSortRunLong ? 0 : kSortLoMax;
    }
    c.kw_used = 2;
    const bool deep = c.hs.tie_big || c.hs.tie_deep;
    const bool tiles_current = !deep && !c.hs.err;
    if (deep) refine_ties(c);
    if (c.hs.err) {
        // more nodes than room: grow before the node phase
        int64_t need = (int64_t)c.hs.n_int + c.hs.nin;
        alloc_nodes(c, need + need / 4 + 64);
        int zero = 0;
        AG2_HIP(hipMemcpy(&c.ds->err, &zero, sizeof(int), hipMemcpyHostToDevice));
    }
    c.nin = c.hs.nin;
    c.n_int = c.hs.n_int;
    // Simulation.cpp:126: the visual-density radius comes from the first tree
    if (c.vd_radius0 == 0.0) c.vd_radius0 = __builtin_bit_cast(double, c.hs.Rbits) / 100000;
    c.n_nodes = c.hs.n_nodes;
    int nin = c.nin, nn = c.n_nodes;
    const NodeArrays o = node_arrays(c);
    if (nn > 0) {
        PVals pv{c.x, c.y, c.z, c.m, c.vx, c.vy, c.vz, c.type};
        // internal nodes with every node's parent and rank, the child-place
        // scan, then node sums, moments and walk records
        int gn = grid_for(nn, 256);
        int nbn = (nn + 1023) / 1024;
        // the leaves and block sums from build_order are stale after a
        // refinement re-ordered the particles or the node arrays grew
        if (nin > 0 && !tiles_current) {
            launch_leaves(c);
            launch_tile_sums(c);
        }
        if (nin == 0) hipLaunchKernelGGL(k_make_root_only, dim3(1), dim3(64), 0, st, o, c.n_bsum);
        else if (c.n_int > 0)
            launch_internal(c, o);
        NodeSums *blk1, *blk2;
        tile_sum_buffers(c, &blk1, &blk2);
        hipLaunchKernelGGL(k_iscan_apply, dim3(nbn), dim3(256), 0, st, nn, c.n_nchild, c.n_bsum, c.n_cstart,
                           (nin + kLevTile - 1) / kLevTile, c.leaf_part, c.ds);
        auto moments = [&](auto per) {
            constexpr int kPer = decltype(per)::value;
            hipLaunchKernelGGL(k_node_moments<kPer>, dim3(grid_for(nn, kPer)), dim3(256), 0, st, nn, nin, n, proot, c.p.split_threshold,
                               c.zero_mass > 0 ? 1 : 0, c.rid, c.ds,
                               c.n_first, c.n_count, c.n_parent, c.n_pidx, c.n_level, blk1, blk2, c.gas_table,
                               c.gas_equal, c.gas_count, pv,
                               c.n_nchild, c.n_rank, c.n_cstart, c.n_gas, c.tnode,
                               c.sph_active ? c.tsph : nullptr, c.g_first, c.g_fired);
        };
        if (nn <= kMomentsSpread) moments(std::integral_constant<int, 64>{});
        else moments(std::integral_constant<int, 256>{});
        c.groups_cleared = true;
        if (deep && nin > 0) {
            // the walk's stack bound comes from the branching depth here
            // (g_list is free until the density phase)
            hipLaunchKernelGGL(k_zero_inner, dim3(gn), dim3(256), 0, st, nn, c.g_list, c.ds);
            hipLaunchKernelGGL(k_count_inner, dim3(gn), dim3(256), 0, st, nn, c.n_pidx, c.n_parent, c.g_list);
            hipLaunchKernelGGL(k_branch_depth, dim3(grid_for(nin, 256)), dim3(256), 0, st, nin, c.base, c.cnt,
                               c.n_parent, c.g_list, c.ds);
            AG2_HIP(hipMemcpyAsync(&c.hs_pinned->walk_depth, &c.ds->walk_depth, sizeof(int32_t),
                                   hipMemcpyDeviceToHost, st));
            AG2_HIP(hipStreamSynchronize(st));
            if (c.hs_pinned->walk_depth > kWalkGrowthMax) {
                c.tree_valid = false;
                throw CapacityError("the walk's stack could grow by " + std::to_string(c.hs_pinned->walk_depth) +
                                    " blocks along one path of this tree, more than it holds (" +
                                    std::to_string(kWalkGrowthMax) + ")");
            }
        }
    }
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[3], st));
    AG2_HIP(hipGetLastError());
    c.tree_valid = true;
}

void build_tree(Ctx &c) {
    build_tree_a(c);
    AG2_HIP(hipEventSynchronize(c.ev_counts));
    build_tree_b(c);
}

}  // namespace ag2
