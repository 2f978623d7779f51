// Barnes-Hut gravity walk with the embedded SPH force:
// Tree::calculateForces (Tree.cpp:57-83) -> Node::calculateGravityForce
// (Node.cpp:247-399) -> Node::calcSPHForce (Node.cpp:88-172).
//
// walk_block: one wavefront per group of 8, 16 or 64 targets (walk_tpg) that are
// consecutive in key order (spatial neighbours).  The wave walks a child-contiguous copy of
// the tree together.  Each iteration pops up to eight sibling blocks (64
// nodes, one per lane) from an LDS stack of (first child, count, lane mask)
// and classifies every node against the group's bounding box:
//   - accepted by every lane of the block's mask -> one batch entry;
//   - opened by every lane of the mask -> its child block is pushed;
//   - mixed -> each target lane runs the reference's own opening test, and
//     ballots give the entry mask (lanes that accept) and the pushed mask
//     (lanes that open).
// Entries and pushes are appended with ballot + mbcnt, so every lane sees
// exactly the node set of its own recursive walk in the reference
// (Node.cpp:382-396 visits the children of an opened node; the visiting order
// differs, which only reorders the sum).  Entries are swept 64 at a time:
// lane j stages entry j in LDS, and each lane computes its interactions with
// the staged entries it belongs to (walk_block: two queues, by lane mask).
// The opening test decides radius^2 against theta^2 r^2 with a 1e-10 margin
// and falls back to the reference's correctly rounded radius / sqrt(r^2)
// inside the margin, so the decision equals the reference's bit for bit.
//
// SPH (the term the reference adds at every accepted gas node within 2 h of
// a gas target): the gravity walk (KIND 1) records, per active gas target,
// the accepted gas nodes within a loose margin of 2 h in a list of kSphK
// node records, going on in spill chunks where a small opening angle accepts
// more; k_sph_pairs then evaluates the lists, eight lanes per target, with the
// exact r < 2 h test and the reference's self skip.  Where the chunks ran out,
// the overflow walk (KIND 2) walks the groups of those targets again with the
// SPH term inline.  Gas-free uploads use
// the KIND 0 kernels, which carry no SPH code.
//
// FP64 sweep: the reference's softened law G m / (r^2 + e0^2) d / r.
// FP32 sweep (split precision): node centres and targets become FP32 offsets
// from the group's bounding-box centre in units of the root half-width
// (FP64 subtraction first), masses are scaled by the root mass, the force
// is m' / sqrt(r'^2 (r'^2 + e'^2)^2) with one v_rsq_f32; a partial chunk, or
// half of a full one, is summed plainly and added to the running total with
// Kahan compensation.
// The SPH term is FP64 in both forms.
#include "ag2_internal.h"
#include "fp64_math.h"

#include <type_traits>

namespace ag2 {
namespace {

constexpr int kWaves = 4;
constexpr int kStackCap = kWalkStackCap;   // pending child blocks per wave
constexpr int kEnt = 128;        // batch entries: < 64 left after a sweep + <= 64 added per iteration
constexpr int kSphK = kSphListLen;   // recorded SPH candidates per gas target (more: spill chunks, then the overflow walk)

// A pending block of siblings: nodes first .. first+count-1, opened by the
// lanes in mask.
struct alignas(16) StackEnt {
    int32_t first, count;
    unsigned long long mask;
};

struct BlockLds {
    StackEnt stk[kStackCap];
    int32_t ent_full[kEnt];              // entries that act on every target (the overflow walk: its pending pairs)
    int32_t ent_node[kEnt];              // entries under a lane mask
    unsigned long long ent_mask[kEnt];
    union {
        double4 d[64];                                        // FP64 sweep: centre and G m
        struct { float4 f[64], lo[64]; } s;                   // FP32 sweep: offsets, their remainders
        double acc[4][64];                                    // SPH sums per target lane; mixed-node staging
    } e;
};
// four workgroups of four waves per CU
static_assert(sizeof(BlockLds) * kWaves * 4 <= 160 * 1024, "the walk's LDS sets its occupancy");

struct WalkArgs {
    int n, nin, nn;
    const core::TreeNode *__restrict__ tree;
    const core::SphNode *__restrict__ tsph;
    // SPH candidate lists: gslot[t] = list slot of key-order target t (-1:
    // none), sph_list[slot * kSphK + k], sph_cnt[slot]; past kSphK candidates a
    // list goes on in spill chunks of kSphK (their numbers in sph_more[slot *
    // kSphMore + ..]; spill_cap chunks, taken with a counter) and sets
    // gover[group of 64]: see list_overflowed
    const int32_t *__restrict__ gslot;
    int32_t *sph_list, *sph_cnt, *sph_spill, *sph_more;
    int spill_cap;
    uint8_t *gover;
    const double *__restrict__ sx, *__restrict__ sy, *__restrict__ sz, *__restrict__ sm;
    const uint8_t *__restrict__ stype;
    const double *__restrict__ svx, *__restrict__ svy, *__restrict__ svz;
    const double *__restrict__ h, *__restrict__ rho, *__restrict__ P;
    const uint8_t *__restrict__ active;
    const DevState *ds;
    unsigned long long *cbins;   // spread counters (bin_add), folded into the DevState after the forces
    core::WalkParams wp;
    double *ax, *ay, *az, *dUdt, *pot;
    DevState *dsw;
    // split-precision walk: near pairs per group (count, then kNearRecs
    // records of node and lane mask), evaluated in FP64 by k_near_pass
    int32_t *near_cnt, *near_node;
    unsigned long long *near_mask;
};

__device__ inline int rl(int v, int j) { return __builtin_amdgcn_readlane(v, j); }
__device__ inline float rl(float v, int j) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j)); }
__device__ inline double uni(double v) {
    long long b = __double_as_longlong(v);
    int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
    int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline float uni(float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); }
__device__ inline double rl(double v, int j) {
    long long b = __double_as_longlong(v);
    int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), j);
    int hi = __builtin_amdgcn_readlane((int)(b >> 32), j);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline unsigned long long rl(unsigned long long v, int j) {
    int lo = __builtin_amdgcn_readlane((int)(v & 0xffffffffull), j);
    int hi = __builtin_amdgcn_readlane((int)(v >> 32), j);
    return ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo;
}
// v_writelane_b32 (the compiler's own intrinsic; clang has no builtin for
// it): lane j of the result is v (uniform), the other lanes keep old.  One
// instruction per dword where a select on lane == j costs a compare, moves
// and selects.
extern "C" __device__ int ag2_writelane_i32(int v, int j, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ inline unsigned long long wl(unsigned long long old, unsigned long long v, int j) {
    const unsigned lo = (unsigned)ag2_writelane_i32((int)(v & 0xffffffffull), j, (int)(old & 0xffffffffull));
    const unsigned hi = (unsigned)ag2_writelane_i32((int)(v >> 32), j, (int)(old >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
__device__ inline int shfl_i(int v, int src) { return __shfl(v, src, 64); }
__device__ inline unsigned long long shfl_u64(unsigned long long v, int src) {
    unsigned lo = (unsigned)__shfl((int)(v & 0xffffffffull), src, 64);
    unsigned hi = (unsigned)__shfl((int)(v >> 32), src, 64);
    return ((unsigned long long)hi << 32) | lo;
}
__device__ inline double shfl_d(double v, int src) {
    long long b = __double_as_longlong(v);
    unsigned lo = (unsigned)__shfl((int)(b & 0xffffffffll), src, 64);
    unsigned hi = (unsigned)__shfl((int)(b >> 32), src, 64);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline void bin_add(unsigned long long *bins, int counter, int bin, unsigned long long v) {
    if (v) atomicAdd(&bins[((size_t)counter * kCountBins + (bin & (kCountBins - 1))) * 8], v);
}

// Number of set bits of b below this lane.
__device__ inline int mbcnt(unsigned long long b) {
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(b >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b, 0u));
}
// Lane-mask -> per-lane bool with no vector work (the mask is the condition).
__device__ inline bool in_mask(unsigned long long m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
// The SPH term with the target's constants hoisted (core::sph_term_hoisted:
// the reference's arithmetic bit for bit).
__device__ inline void sph_pair(double dx, double dy, double dz, double r2, double gas, double vx, double vy,
                                double vz, const core::SphConst &k, core::WalkSums *s) {
    core::sph_term_hoisted(dx, dy, dz, r2, gas, vx, vy, vz, k, s);
}

// The same term, value for value, with the square root and the four quotients
// in short correctly rounded forms: one estimate and its Newton steps serve
// the root and the quotient by r (Goldschmidt's iteration, two corrections by
// the root's remainder), 1 / h (ih) is formed once per target, and each
// quotient ends with one step on its exact remainder (Markstein).  The compiler's
// general forms scale their operands against overflow and fix up special
// values on every call; plain_support and plain_pair stand for that here
// (every intermediate and remainder far inside the normal range), and what
// lies outside takes sph_pair.  Compared with / and sqrt over 2e8 random
// operands, the estimates off by their full 5.3e-8: no result differs.
__device__ inline bool plain_support(double h) { return h > 0x1p-100 && h < 0x1p100; }

// r2 = |d|^2 > 0, vd = v . d, hv = h vd (which the term divides where vd < 0)
__device__ inline bool plain_pair(double r2, double vd, double hv) {
    return r2 > 0x1p-300 && !(vd < 0.0 && !(hv < -0x1p-500 && hv > -0x1p500));
}

// sqrt(x), and 1 / sqrt(x) to the last bit or so.
__device__ inline double root_plain(double x, double *inv) {
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, hy = 0.5 * y;
    const double e = __builtin_fma(-hy, g, 0.5);
    hy = __builtin_fma(hy, e, hy);
    g = __builtin_fma(g, e, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), hy, g);
    g = __builtin_fma(__builtin_fma(-g, g, x), hy, g);
    const double i = hy + hy;
    *inv = __builtin_fma(__builtin_fma(-g, i, 1.0), i, i);
    return g;
}

// a / b from y = 1 / b.
__device__ inline double quot_plain(double a, double b, double y) {
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}

// The term of a pair within 2 h: r = sqrt(r2), ir = 1 / r.
__device__ inline void sph_pair_plain(double dx, double dy, double dz, double r, double ir, double gas, double vx,
                                      double vy, double vz, double vd, double hv, const core::SphConst &k, double ih,
                                      double *sx, double *sy, double *sz, double *su) {
    const double q = quot_plain(r, k.h, ih);
    const double near = -3.0 * q + 2.25 * q * q, far = -0.75 * ((2 - q) * (2 - q));
    const double poly = q < 1.0 ? near : far;
    const double gsc = quot_plain(quot_plain(k.a3 * poly, k.h, ih), r, ir);
    const double gx = dx * gsc, gy = dy * gsc, gz = dz * gsc;
    const double den = r * r + k.eta_h2;
    double z = __builtin_amdgcn_rcp(den);
    z = __builtin_fma(__builtin_fma(-den, z, 1.0), z, z);
    z = __builtin_fma(__builtin_fma(-den, z, 1.0), z, z);
    const double mu = quot_plain(hv, den, z);
    const double MU = vd < 0 ? -0.5 * k.cij * mu + 1.0 * (mu * mu) : 0.0;
    const double fp = -gas * k.pr, fv = -gas * MU;
    double ax = fp * gx, ay = fp * gy, az = fp * gz;
    ax += fv * gx;
    ay += fv * gy;
    az += fv * gz;
    *su += 0.5 * gas * (k.pr + MU) * (vx * gx + vy * gy + vz * gz);
    const bool bad = ax != ax || ay != ay || az != az;
    if (__any(bad)) {
        ax = bad ? 0.0 : ax;
        ay = bad ? 0.0 : ay;
        az = bad ? 0.0 : az;
    }
    *sx += ax; *sy += ay; *sz += az;
}

// Workgroups reach the 8 XCDs round robin.  Neighbouring groups read mostly
// the same tree records and should share one XCD's L2, but one contiguous
// eighth of the key order per XCD leaves XCDs idle behind the one that holds
// the longest lists.  So each XCD takes runs of kXcdRun workgroups in turn
// (the last, incomplete round is split evenly).  Walk kernel, one eighth per
// XCD / runs of 16: 1 M disk FP32 755 / 709 us, FP64 1,242 / 1,192; 1 M
// Hernquist 669 / 620; 100,003 disk 158 / 143; 2 M 1,370 / 1,315; 200,000
// 241 / 244; 3 M 1,947 / 1,966.  Runs of 2, 4, 8 and 32 lie between; of 64,
// 720 us at 1 M.
constexpr int kXcdRun = 16;
__device__ inline int walk_workgroup(int b, int nb) {
    const int whole = nb / (8 * kXcdRun) * (8 * kXcdRun);
    if (b >= whole) return whole + xcd_block(b - whole, nb - whole);
    const int x = b & 7, i = b >> 3;
    return (i / kXcdRun * 8 + x) * kXcdRun + i % kXcdRun;
}

// Transpose of a 64 x 64 bit matrix held one row per lane: lane j gives row j
// (lo: columns 0..31, hi: 32..63) and gets column j.  Halves are exchanged
// at lane distance 32, 16, .. 1, on the vector unit alone (30 instructions).
__device__ inline void transpose64(unsigned &lo, unsigned &hi) {
    const int lane = lane_id();
    auto s32 = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
    const unsigned a = s32[0], b = s32[1];
    // 16: both words' low halves in one register, their high halves in another
    auto s16 = __builtin_amdgcn_permlane16_swap(__builtin_amdgcn_perm(b, a, 0x05040100),
                                                __builtin_amdgcn_perm(b, a, 0x07060302), false, false);
    unsigned w[2] = {__builtin_amdgcn_perm(s16[1], s16[0], 0x05040100),
                     __builtin_amdgcn_perm(s16[1], s16[0], 0x07060302)};
    const unsigned sel8 = (lane & 8) ? 0x03070105u : 0x06020400u;
    const unsigned m4 = (lane & 4) ? 0xf0f0f0f0u : 0x0f0f0f0fu, r4 = (lane & 4) ? 4u : 28u;
    const unsigned m2 = (lane & 2) ? 0xccccccccu : 0x33333333u, r2 = (lane & 2) ? 2u : 30u;
    const unsigned m1 = (lane & 1) ? 0xaaaaaaaau : 0x55555555u, r1 = (lane & 1) ? 1u : 31u;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        unsigned v = w[k], y;
        y = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true);   // lane ^ 8 (row_ror:8)
        v = __builtin_amdgcn_perm(y, v, sel8);
        y = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, true);   // lane ^ 7 (row_half_mirror)
        y = (unsigned)__builtin_amdgcn_mov_dpp((int)y, 0x1b, 0xf, 0xf, true);    // lane ^ 4
        v = (v & m4) | (__builtin_amdgcn_alignbit(y, y, r4) & ~m4);
        y = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, true);    // lane ^ 2
        v = (v & m2) | (__builtin_amdgcn_alignbit(y, y, r2) & ~m2);
        y = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true);    // lane ^ 1
        v = (v & m1) | (__builtin_amdgcn_alignbit(y, y, r1) & ~m1);
        w[k] = v;
    }
    lo = w[0];
    hi = w[1];
}

// The set bits of m in ascending order, two at a time: f(j1, j2, both); j2 is
// j1 again where m has no second bit.  Two entries' loads and arithmetic
// overlap: one at a time, every pass waits out a chain of about twenty
// dependent instructions behind an LDS read.
template <class F>
__device__ __forceinline__ void bit_pairs(unsigned m, F &&f) {
    while (m) {
        const int j1 = __builtin_ctz(m);
        m &= m - 1;
        const bool both = m != 0;
        const int j2 = both ? __builtin_ctz(m) : j1;
        m &= m - 1;
        f(j1, j2, both);
    }
}

// Is a target with cnt candidates left to the overflow walk?  When the spill
// chunks ran out, every target past its list is, so that which of them got a
// chunk (a matter of timing) decides nothing.
__device__ inline bool list_overflowed(const WalkArgs &a, int cnt) {
    return cnt > kSphK * (1 + kSphMore) || (cnt > kSphK && (a.spill_cap == 0 || a.ds->spill_next > a.spill_cap));
}

// Group g of TPG targets: particles TPG g .. TPG g + TPG - 1 in key order.
// KIND 0: gravity.  KIND 1: gravity, and every accepted gas node within a
// margin of 2h of a gas target goes on that target's SPH candidate list
// (evaluated by k_sph_pairs).  KIND 3: FP64 gravity again for the groups whose
// split-precision walk found more near pairs than kNearRecs (their results
// replace that walk's).  KIND 2: the SPH term, inline, for the targets
// whose list overflowed (groups flagged in gover only; no gravity).
// KIND 4: the FP64 potential of every target (active or not).
//
// TPG < 64: lane l works for target l % TPG; the NS = 64 / TPG lanes of a
// target split the opening tests of mixed nodes and the swept entries among
// them (lane masks of nodes and entries have TPG bits).  See walk_tpg for
// the choice.
//
// An accepted node becomes an entry of one of two queues, each swept 64
// entries at a time:
//  - full: every target of the group interacts and none is near; the sweep
//    has no lane mask at all (a fifth to a third of the entries);
//  - partial: the 64 lane masks are transposed (transpose64), and each lane
//    walks the bits of its own word, entry by entry, reading the entry from
//    LDS.  The loop ends with the busiest lane: on the 1 M disk the partial
//    masks hold a fifth of the lanes on average, and a lane meets at most
//    two fifths of a chunk, where a sweep under the masks ran over all of it.
// The walk is bound by VALU issue (82 % of the SIMDs' cycles): with the two
// queues, the SPH margin tested in the sweep and two entries in flight per
// lane it issues 22.4 k vector instructions per wave where one masked sweep
// issued 28.4 k (1 M disk, FP32), and the kernel takes 0.69 ms against
// 1.00 ms; the FP64 form 1.00 ms against 1.90 ms.
template <bool F32, int KIND, int TPG>
__device__ __forceinline__ void walk_block(const WalkArgs &a, int g, BlockLds *lds) {
    static_assert(TPG == 64 || TPG == 16 || TPG == 8, "targets per group");
    static_assert(KIND != 2 || TPG == 64, "overflow flags are per group of 64 targets");
    constexpr int NS = 64 / TPG;
    constexpr unsigned long long kAll = TPG == 64 ? ~0ull : (1ull << (TPG & 63)) - 1;
    constexpr bool GAS = KIND == 1 || KIND == 2;
    if (g >= (a.n + TPG - 1) / TPG) return;
    if (KIND == 2 && !a.gover[g]) return;
    if (KIND == 3 && a.near_cnt[g] <= kNearRecs) return;
    const int wv = threadIdx.x >> 6;
    const int lane = lane_id();
    BlockLds &S = lds[wv];
    const int tl = lane & (TPG - 1), sub = lane / TPG;
    const int t = g * TPG + tl;
    const bool valid_t = t < a.n;
    const int q = t;   // particle state is in key order
    const bool act = valid_t && (KIND == 4 || a.active[q] != 0);
    double px = 0.0, py = 0.0, pz = 0.0, pm = 0.0;
    if (valid_t) {
        px = a.sx[t]; py = a.sy[t]; pz = a.sz[t]; pm = a.sm[t];
    }
    const bool tgas = valid_t && a.stype[t] == 2;
    const double th = KIND != 4 && act ? a.h[q] : 0.0;
    const unsigned long long amask = __ballot(act && pm != 0.0) & kAll;
    const bool mine = (amask >> tl) & 1ull;
    bool sph_lane = GAS && mine && tgas && th > 0.0;
    int slot = -1;
    if (GAS && sph_lane) {
        slot = a.gslot[t];
        if (KIND == 2) sph_lane = list_overflowed(a, a.sph_cnt[slot]);
    }
    const unsigned long long sphB = __ballot(sph_lane);   // all NS lanes of a target
    if (KIND == 2 && !sphB) return;
    const double h2x4 = GAS ? (2.0 * th) * (2.0 * th) : 0.0;   // SPH support (2h)^2
    int lcnt = 0;   // KIND 1: candidates recorded for this target

    core::WalkSums s{0, 0, 0, 0, 0, 0, 0};
    unsigned long long nint = 0ull;   // uniform: interactions of the whole wave
    double invL = 0.0, invMu = 0.0;
    float xr = 0.f, yr = 0.f, zr = 0.f, e2f = 0.f;
    float xlo = 0.f, ylo = 0.f, zlo = 0.f;   // FP32 remainders of the target offsets (near chunks)
    float r2df = 0.f;                         // near chunks: r^2 below which the pair goes to the FP64 pass
    // FP32 form: entries closer than r2min (scaled units) to this lane's
    // target are too close for FP32 offsets to resolve their direction; they
    // are recorded and evaluated in FP64 after the walk (k_near_pass)
    float r2min = 0.f;
    double near_b2 = 0.0;   // uniform: see the full-queue test
    unsigned lnint = 0u;    // interactions counted per lane
    int nrec = 0;           // uniform: near pairs recorded for k_near_pass
    bool dfmode = false;    // uniform: this group's chunks carry the offsets' remainders
    float sumx = 0.f, sumy = 0.f, sumz = 0.f, cmpx = 0.f, cmpy = 0.f, cmpz = 0.f;
    const double theta = a.wp.theta, th2 = a.wp.theta * a.wp.theta;
    const double th2lo = th2 * (1.0 - 1e-10), th2hi = th2 * (1.0 + 1e-10);   // group-box accept / open margins
    const double inv_th2m = 1.0 / (th2 * (1.0 - 1e-10));         // mixed-node accept threshold factor
    const double open_ratio = (1.0 - 1e-10) / (1.0 + 1e-10);     // open threshold / accept threshold
    const double e02 = a.wp.e0 * a.wp.e0;
    const double R = __longlong_as_double((long long)a.ds->Rbits);

    if (amask != 0ull && a.nn > 0) {
        // bounding box of the group's active targets (decides whole-group
        // accept / open for most nodes without per-lane tests)
        double lo[3] = {px, py, pz}, hi[3] = {px, py, pz};
        if (!mine) { lo[0] = lo[1] = lo[2] = 1e308; hi[0] = hi[1] = hi[2] = -1e308; }
        // box of the SPH targets and their largest support 2h
        double glo[3] = {px, py, pz}, ghi[3] = {px, py, pz}, h2 = sph_lane ? 2.0 * th : 0.0;
        if (!sph_lane) { glo[0] = glo[1] = glo[2] = 1e308; ghi[0] = ghi[1] = ghi[2] = -1e308; }
        for (int d = TPG / 2; d >= 1; d >>= 1) {
            for (int k = 0; k < 3; k++) {
                double a1 = __shfl_xor(lo[k], d, 64), b1 = __shfl_xor(hi[k], d, 64);
                lo[k] = a1 < lo[k] ? a1 : lo[k];
                hi[k] = b1 > hi[k] ? b1 : hi[k];
            }
            if (sphB) {
                for (int k = 0; k < 3; k++) {
                    double a1 = __shfl_xor(glo[k], d, 64), b1 = __shfl_xor(ghi[k], d, 64);
                    glo[k] = a1 < glo[k] ? a1 : glo[k];
                    ghi[k] = b1 > ghi[k] ? b1 : ghi[k];
                }
                double c1 = __shfl_xor(h2, d, 64);
                h2 = c1 > h2 ? c1 : h2;
            }
        }
        for (int k = 0; k < 3; k++) {
            lo[k] = uni(lo[k]); hi[k] = uni(hi[k]); glo[k] = uni(glo[k]); ghi[k] = uni(ghi[k]);
        }
        const double reach2 = uni(h2 * h2) * (1.0 + 1e-9);
        const double gcx = 0.5 * (lo[0] + hi[0]), gcy = 0.5 * (lo[1] + hi[1]), gcz = 0.5 * (lo[2] + hi[2]);
        if (F32) {
            double Mu = a.tree[0].mass;
            invL = uni(R > 0 ? 1.0 / R : 1.0);
            invMu = uni(Mu > 0 ? 1.0 / Mu : 1.0);
            const double oxd = (px - gcx) * invL, oyd = (py - gcy) * invL, ozd = (pz - gcz) * invL;
            xr = (float)oxd; yr = (float)oyd; zr = (float)ozd;
            xlo = (float)(oxd - (double)xr); ylo = (float)(oyd - (double)yr); zlo = (float)(ozd - (double)zr);
            double el = a.wp.e0 * invL;
            e2f = uni((float)(el * el));
            // each offset is rounded to 2^-24 of itself, so d carries an error
            // of about 2^-24 (|target| + |entry|) per component; below 2^-8
            // of 2 (|x| + |y| + |z|) of the target offset the FP32 direction
            // could be off by more than 2^-15, and FP32 may round d to zero
            // where the FP64 positions differ (the reference's r == 0 skip is
            // on FP64 r)
            // (and a pair needs r^2 (r^2 + e^2)^2 in v_rsq_f32's normal range:
            // below the floor a group far smaller than the softening length
            // leaves it)
            const double fl = 0x1p-123 / ((double)e2f * (double)e2f);
            const float floor2 = uni((float)(fl < 0x1p-41 ? fl : 0x1p-41));
            const float off = 2.f * (fabsf(xr) + fabsf(yr) + fabsf(zr));
            r2min = fmaxf(off * off * 0x1p-16f, floor2);
            const float ao = sqrtf(r2min);
            // in a chunk with such an entry the sweep forms d from the offsets
            // and their remainders (48 bits: exact difference of the high parts
            // for close pairs by Sterbenz), which resolves the direction down
            // to 2^-34 of the offsets; closer pairs go to the FP64 pass
            const float adf = off * 0x1p-34f;
            r2df = fmaxf(adf * adf, floor2);
            // an entry at distance D from the targets' box, beyond near_a +
            // 2^-20 of its offset sum, is beyond every lane's r2min with room
            // for the FP32 offsets' rounding (2^-23 of target and entry
            // offsets), so its lanes need no per-lane test.  The offset sum is
            // at most ext + sqrt(3) D, so D (1 - 2^-19) > near_a + 2^-20 ext
            // is enough.
            float aomax = mine ? ao : 0.f;
            for (int d = TPG / 2; d >= 1; d >>= 1) aomax = fmaxf(aomax, __shfl_xor(aomax, d, 64));
            const double ext = 0.5 * ((hi[0] - lo[0]) + (hi[1] - lo[1]) + (hi[2] - lo[2])) * invL;
            const double near_a = uni(4.0 * (double)aomax + 0x1p-20 * ext);
            const double nb = (near_a + 0x1p-20 * ext) * (1.0 + 0x1p-18) * R;
            near_b2 = nb * nb;
        }
        // KIND 1: the candidate test on the sweep's own r^2, loose by a
        // margin; k_sph_pairs decides exactly.  In the split form r is
        // computed from FP32 offsets from the group centre, each rounded by at
        // most 2^-24 of its size: for a node within 2h (scaled: D) of a target
        // with offset sum A, the computed r exceeds the true one by less than
        // 2^-23 (A + D) + rounding of r^2 itself.
        const double lim64 = sph_lane ? h2x4 * (1.0 + 1e-9) : -1.0;
        float lim32 = 0.f;
        if (F32 && KIND == 1) {
            const double D = 2.0 * th * invL;
            const double A = fabs((double)xr) + fabs((double)yr) + fabs((double)zr);
            const double rl32 = D * (1.0 + 1e-6) + 2.4e-7 * (A + 2.0 * D);
            lim32 = sph_lane ? (float)(rl32 * rl32 * (1.0 + 1e-5)) : -1.f;
        }
        int32_t *lbase = (KIND == 1 && slot >= 0) ? a.sph_list + (size_t)slot * kSphK : nullptr;   // current chunk
        // Multi-block pops keep the stack within kStackCap: a pop of up to
        // 64 nodes pushes at most 64 blocks, and above `single_above` the walk
        // pops one block at a time; from any point the stack then grows by at
        // most walk_depth blocks (7 per level below, or in a deep tree the
        // sum of (internal children - 1) along a path -- leaves and bucket
        // members push nothing).  The build refuses trees where that bound
        // exceeds kStackCap - 1.
        const int growth = __builtin_amdgcn_readfirstlane(a.ds->walk_depth);
        const int single_above = kStackCap - 64 - growth;
        if (lane == 0) { S.stk[0].first = 0; S.stk[0].count = 1; S.stk[0].mask = amask; }
        int sp = 1;
        int nf = 0, ni = 0;   // full and partial entries queued
        unsigned long long n_entries = 0ull, n_tests = 0ull, n_mixed = 0ull;
        while (true) {
            wave_sync_lds();
            if (sp > 0) {
                // ------------------------------------------- pop blocks
                int k = sp > single_above ? 1 : (sp < 8 ? sp : 8);
                StackEnt se{0, 0, 0ull};
                if (lane < k) se = S.stk[sp - 1 - lane];
                // (lanes at or past k hold count 0.)  The ballots of the pop
                // are of plain compares, combined on the scalar unit: a ballot
                // of a bool formed across a divergent branch costs a select
                // and a compare to rebuild its mask.
                const unsigned long long big = __ballot(se.count > 8);
                if (big) k = __builtin_ctzll(big) + 1;   // a bucket block is taken 8 at a time
                const int b = lane >> 3, sl = lane & 7;
                const int fb = shfl_i(se.first, b), cb = shfl_i(se.count, b);
                const unsigned long long Mb = shfl_u64(se.mask, b);
                sp -= k;
                if (big) {
                    if (lane == k - 1) { S.stk[sp].first = se.first + 8; S.stk[sp].count = se.count - 8; S.stk[sp].mask = se.mask; }
                    sp++;
                }
                const unsigned long long validB = __ballot(b < k) & __ballot(sl < cb);
                const int node = fb + sl;
                // lane classifies its node against the group box: 1 accept
                // for every lane, 2 open for every lane, 3 decide per lane,
                // 0 nothing (no node or mass 0)
                core::TreeNode r;
                int cls = 0, rnch = 0, rpidx = -1;
                double rad = 0.0, rmin2 = 0.0;
                if (in_mask(validB)) {
                    r = a.tree[node];
                    rnch = r.nchild;
                    rpidx = r.pidx;
                    rad = ldexp(R, -(int)r.level);
                    // nearest and farthest box points from the centre;
                    // the 1e-10 margins absorb the fused roundings
                    const double ax = lo[0] - r.cx, bx = r.cx - hi[0];
                    const double ay = lo[1] - r.cy, by = r.cy - hi[1];
                    const double az = lo[2] - r.cz, bz = r.cz - hi[2];
                    const double ex = fmax(fmax(ax, bx), 0.0), ey = fmax(fmax(ay, by), 0.0), ez = fmax(fmax(az, bz), 0.0);
                    rmin2 = __builtin_fma(ex, ex, __builtin_fma(ey, ey, ez * ez));
                    if (r.mass == 0.0) cls = 0;
                    else if (r.pidx >= 0) cls = 1;
                    else {
                        const double fx = fmax(fabs(ax), fabs(bx)), fy = fmax(fabs(ay), fabs(by)), fz = fmax(fabs(az), fabs(bz));
                        const double rmax2 = __builtin_fma(fx, fx, __builtin_fma(fy, fy, fz * fz));
                        const double rad2 = rad * rad;
                        if (rmin2 > 0.0 && rad2 < th2lo * rmin2) cls = 1;
                        else if (rmin2 > 0.0 && rad2 > th2hi * rmax2) cls = 2;
                        else cls = 3;
                    }
                }
                n_tests += (unsigned long long)__builtin_popcountll(validB);
                // whole-mask accepts -> entries (a leaf never acts on itself:
                // r == 0, Node.cpp:274-276, so only distinct particles reach
                // the sweeps' r == 0 and near-pair tests)
                const unsigned long long c1B = __ballot(cls == 1);
                const int self = rpidx - g * TPG;
                const bool drop = rpidx >= 0 && (unsigned)self < (unsigned)TPG;   // (its own leaf: a leaf is class 1 or 0)
                const unsigned long long A = drop ? Mb & ~(1ull << (self & 63)) : Mb;
                const unsigned long long appB = c1B & __ballot(A != 0ull);
                unsigned long long fullB = 0ull;
                if (KIND != 2) {
                    fullB = appB & __ballot(A == amask);
                    if (F32) fullB &= __ballot(rmin2 > near_b2);
                    if (in_mask(fullB)) S.ent_full[nf + mbcnt(fullB)] = node;
                    nf += __builtin_popcountll(fullB);
                }
                const unsigned long long partB = appB & ~fullB;
                if (in_mask(partB)) {
                    const int slot = ni + mbcnt(partB);
                    S.ent_node[slot] = node;
                    S.ent_mask[slot] = A;
                }
                ni += __builtin_popcountll(partB);
                // whole-mask opens -> child blocks
                const unsigned long long nchB = __ballot(rnch > 0);
                const unsigned long long pB = __ballot(cls == 2) & nchB;
                if (in_mask(pB)) {
                    const int slot = sp + mbcnt(pB);
                    if (slot < kStackCap) {
                        S.stk[slot].first = r.first_child; S.stk[slot].count = r.nchild; S.stk[slot].mask = Mb;
                    } else {
                        a.dsw->walk_err = 1;   // unreachable: see single_above
                    }
                }
                sp += __builtin_popcountll(pB);
                if (sp > kStackCap) sp = kStackCap;
                // per-lane decisions, exactly the reference's test
                const unsigned long long mixB = __ballot(cls == 3);
                if (mixB) {
                    const int nmix = __builtin_popcountll(mixB);
                    n_mixed += (unsigned long long)nmix;
                    // The mixed nodes' centres and thresholds go to the staging
                    // area (free outside the sweep) and are read back NS at a
                    // time, one per NS'th of the wave.  A lane accepts a mixed
                    // node when r^2 > rad^2 / (theta^2 (1 - 1e-10)) and opens
                    // it when r^2 < rad^2 / (theta^2 (1 + 1e-10)): outside
                    // that band the reference's rounded radius / sqrt(r^2) <
                    // theta cannot decide otherwise; inside it, its own
                    // expression decides on its own unfused r^2.  (A centre
                    // that is NaN is never accepted.)  Each node's accept and
                    // open masks are selected into the lane that holds the
                    // node, and its entry and child block are appended after
                    // the loop in lane order.
                    const double tacc = rad * rad * inv_th2m;
                    const int rank = mbcnt(mixB);
                    if (cls == 3) {
                        S.e.acc[0][rank] = r.cx; S.e.acc[1][rank] = r.cy; S.e.acc[2][rank] = r.cz; S.e.acc[3][rank] = tacc;
                    }
                    wave_sync_lds();
                    unsigned long long mAA = 0ull, mOO = 0ull;   // decisions on this lane's mixed node
                    unsigned long long bb = mixB;
                    for (int m0 = 0; m0 < nmix; m0 += NS) {
                        const int at = m0 + sub < nmix ? m0 + sub : nmix - 1;
                        const double ncx = S.e.acc[0][at], ncy = S.e.acc[1][at], ncz = S.e.acc[2][at], Tacc = S.e.acc[3][at];
                        const double dx = ncx - px, dy = ncy - py, dz = ncz - pz;
                        const double r2f = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
                        const unsigned long long nz = __ballot(r2f != 0.0);
                        const unsigned long long ge = __ballot(r2f >= Tacc * open_ratio);
                        unsigned long long AA = __ballot(r2f > Tacc);
                        unsigned long long OO = nz & ~ge;
                        const unsigned long long band = ge & ~AA;
                        if (band) {
                            // the half-widths of the nodes decided here, from their lanes
                            unsigned long long mm = bb;
                            if (TPG < 64) {
                                mm = mixB;
                                for (int u = 0; u < at; u++) mm &= mm - 1;
                            }
                            const double nrad = shfl_d(rad, __builtin_ctzll(mm));
                            const double r2 = dx * dx + dy * dy + dz * dz;
                            const unsigned long long BA = band & __ballot((nrad / sqrt(r2)) < theta);
                            AA |= BA;
                            OO |= band & ~BA;
                        }
                        if (TPG == 64) {
                            const int kk = __builtin_ctzll(bb);
                            bb &= bb - 1;
                            mAA = wl(mAA, AA, kk);
                            mOO = wl(mOO, OO, kk);
                        } else if (cls == 3 && rank - m0 >= 0 && rank - m0 < NS) {
                            mAA = AA >> (TPG * (rank - m0));
                            mOO = OO >> (TPG * (rank - m0));
                        }
                    }
                    mAA &= Mb & kAll;
                    mOO &= Mb & kAll;
                    const unsigned long long eB = mixB & __ballot(mAA != 0ull);
                    if (in_mask(eB)) {
                        const int slot = ni + mbcnt(eB);
                        S.ent_node[slot] = node;
                        S.ent_mask[slot] = mAA;
                    }
                    ni += __builtin_popcountll(eB);
                    const unsigned long long qB = mixB & __ballot(mOO != 0ull) & nchB;
                    if (in_mask(qB)) {
                        const int slot = sp + mbcnt(qB);
                        if (slot < kStackCap) {
                            S.stk[slot].first = r.first_child; S.stk[slot].count = r.nchild; S.stk[slot].mask = mOO;
                        } else {
                            a.dsw->walk_err = 1;
                        }
                    }
                    sp += __builtin_popcountll(qB);
                    if (sp > kStackCap) sp = kStackCap;
                }
            }
            // ------------------------------------------------- sweep
            while (ni >= 64 || nf >= 64 || (sp == 0 && ni + nf > 0)) {
                const bool part = ni >= 64 || (nf < 64 && ni > 0);   // uniform
                const int have = part ? ni : nf;
                const int cnt = have >= 64 ? 64 : have;
                const int e0 = have - cnt;
                const int32_t *enode = part ? S.ent_node : S.ent_full;
                wave_sync_lds();
                double ecx = 0.0, ecy = 0.0, ecz = 0.0;
                // the staged entry's lane mask; TPG < 64: in the field of the
                // sub that sweeps it (entries [TPG s, TPG (s + 1)) of a
                // partial chunk)
                unsigned long long emask = 0ull;
                bool cand = false;
                if (lane < cnt) {
                    const core::TreeNode w = a.tree[enode[e0 + lane]];
                    emask = part ? S.ent_mask[e0 + lane] : amask;
                    if (KIND == 2) { ecx = w.cx; ecy = w.cy; ecz = w.cz; }
                    if (F32) {
                        const double exd = (w.cx - gcx) * invL, eyd = (w.cy - gcy) * invL, ezd = (w.cz - gcz) * invL;
                        S.e.s.f[lane] = make_float4((float)exd, (float)eyd, (float)ezd, (float)(w.mass * invMu));
                        lnint += (unsigned)__builtin_popcountll(emask);   // less the lanes excluded below
                    } else if (KIND != 2) {
                        // G m staged once per entry (the sweep forms ((G m) rcp) ri, as before)
                        S.e.d[lane] = make_double4(w.cx, w.cy, w.cz, KIND == 4 || a.wp.soft_live ? w.mass : a.wp.G * w.mass);
                    }
                    if (GAS && sphB && (emask & sphB)) {
                        // a leaf's gas mass is its mass when it is gas; nodes of
                        // mass 0 never become entries
                        const bool gasn = w.gas > 0.0;
                        double ex = fmax(fmax(glo[0] - w.cx, w.cx - ghi[0]), 0.0);
                        double ey = fmax(fmax(glo[1] - w.cy, w.cy - ghi[1]), 0.0);
                        double ez = fmax(fmax(glo[2] - w.cz, w.cz - ghi[2]), 0.0);
                        cand = gasn && ex * ex + ey * ey + ez * ez < reach2;
                    }
                    if (TPG < 64) emask <<= TPG * (lane / TPG);
                }
                const unsigned long long candB = GAS ? __ballot(cand) : 0ull;
                wave_sync_lds();
                unsigned tlo = (unsigned)emask, thi = (unsigned)(emask >> 32);
                if (KIND != 2 && part) transpose64(tlo, thi);
                // Each half of a lane's word is walked by itself (TPG < 64:
                // only one half holds bits).
                constexpr int kHalves = TPG == 64 ? 2 : 1;
                const int half0 = TPG == 64 ? 0 : (2 * sub) / NS;
                unsigned word[kHalves];
                if (part) {
                    word[0] = half0 ? thi : tlo;
                    if (kHalves == 2) word[kHalves - 1] = thi;
                } else {   // a full chunk: every entry of the lane's field
                    unsigned long long all = (cnt == 64 ? ~0ull : (1ull << cnt) - 1) & (kAll << (TPG * sub & 63));
                    if (!mine) all = 0ull;
                    word[0] = (unsigned)(all >> (32 * half0));
                    if (kHalves == 2) word[kHalves - 1] = (unsigned)(all >> 32);
                }
                // KIND 1: the entries of each half within the lane's SPH
                // margin, as the sweep meets them (the r^2 it has anyway; one
                // compare, select and or per entry, where testing the
                // candidate entries again after the sweep, all lanes at once,
                // was a quarter of the walk's instructions), and the entries
                // resolved or recorded after it
                const bool spot = KIND == 1 && candB != 0ull;   // uniform
                unsigned hit[kHalves] = {};
                unsigned long long hb = 0ull;
                const bool dfc = F32 && dfmode;
                if (KIND == 2) {
                    // no gravity
                } else if (F32) {
                    // Three sweeps, counted from the masks at staging:
                    //  - full: every lane interacts (r2 > r2min > 0 for each), under
                    //    no mask, lanes whose target takes no part included;
                    //  - partial: lanes within r2min of an entry (FP32
                    //    offsets cannot resolve the direction) are left out;
                    //  - dfmode (a group that has met such lanes, every later
                    //    chunk): offsets with their FP32 remainders (48 bits; the
                    //    difference of the high parts is exact for close pairs),
                    //    down to r2df.
                    // Left-out lanes are found again after the sweep: resolved
                    // with the remainders where they can be, else recorded for
                    // the FP64 pass (and dropped from the count).
                    const float4 *fs = S.e.s.f, *fl = S.e.s.lo;
                    float cx = 0.f, cy = 0.f, cz = 0.f;
                    auto pull = [&](float m, float dx, float dy, float dz, float r2, bool ok) {
                        const float s2 = r2 + e2f;
                        float f = m * __builtin_amdgcn_rsqf(r2 * s2 * s2);
                        f = ok ? f : 0.f;
                        cx = __builtin_fmaf(f, dx, cx);
                        cy = __builtin_fmaf(f, dy, cy);
                        cz = __builtin_fmaf(f, dz, cz);
                    };
                    // the plain sums so far to the compensated ones
                    auto settle = [&]() {
                        float y = cx - cmpx, tt = sumx + y; cmpx = (tt - sumx) - y; sumx = tt;
                        y = cy - cmpy; tt = sumy + y; cmpy = (tt - sumy) - y; sumy = tt;
                        y = cz - cmpz; tt = sumz + y; cmpz = (tt - sumz) - y; sumz = tt;
                        cx = cy = cz = 0.f;
                    };
                    int left = 0;   // this lane was left out of some entry
                    if (dfc) {
                        if (lane < cnt) {
                            const core::TreeNode w = a.tree[enode[e0 + lane]];
                            const double exd = (w.cx - gcx) * invL, eyd = (w.cy - gcy) * invL, ezd = (w.cz - gcz) * invL;
                            S.e.s.lo[lane] = make_float4((float)(exd - (double)(float)exd), (float)(eyd - (double)(float)eyd),
                                                         (float)(ezd - (double)(float)ezd), 0.f);
                        }
                        wave_sync_lds();
                        for (int h = 0; h < kHalves; h++) {
                            auto one = [&](int j, bool on) {
                                const float4 e = fs[32 * (half0 + h) + j], l = fl[32 * (half0 + h) + j];
                                const float dx = (e.x - xr) + (l.x - xlo), dy = (e.y - yr) + (l.y - ylo);
                                const float dz = (e.z - zr) + (l.z - zlo);
                                const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                                const bool ok = r2 > r2df;
                                left = ok ? left : 1;   // (a second entry that is the first again changes nothing)
                                pull(e.w, dx, dy, dz, r2, ok && on);
                                if (KIND == 1) hit[h] |= ok && r2 < lim32 ? 1u << j : 0u;
                            };
                            bit_pairs(word[h], [&](int j1, int j2, bool both) { one(j1, true); one(j2, both); });
                        }
                    } else if (part) {
                        // every lane's entries first, with the least r^2 met; a
                        // chunk in which some lane met one within r2min (or no
                        // number at all) is swept again with those left out.
                        // (A compare and two selects per entry the other way:
                        // the 1 M disk's walk 706 us, now 692; 4 M 2,567, now
                        // 2,480.)
                        float least = 3e38f;
                        auto sweep = [&](auto spotting, auto checked) {
                            for (int h = 0; h < kHalves; h++) {
                                hit[h] = 0u;
                                bit_pairs(word[h], [&](int j1, int j2, bool both) {
                                    const float4 e1 = fs[32 * (half0 + h) + j1], e2 = fs[32 * (half0 + h) + j2];
                                    const float dx1 = e1.x - xr, dy1 = e1.y - yr, dz1 = e1.z - zr;
                                    const float dx2 = e2.x - xr, dy2 = e2.y - yr, dz2 = e2.z - zr;
                                    const float q1 = __builtin_fmaf(dx1, dx1, __builtin_fmaf(dy1, dy1, dz1 * dz1));
                                    const float q2 = __builtin_fmaf(dx2, dx2, __builtin_fmaf(dy2, dy2, dz2 * dz2));
                                    if (decltype(checked)::value) {
                                        const bool ok1 = q1 > r2min, ok2 = q2 > r2min;
                                        left = ok1 && ok2 ? left : 1;
                                        pull(e1.w, dx1, dy1, dz1, q1, ok1);
                                        pull(e2.w, dx2, dy2, dz2, q2, ok2 && both);
                                        if (decltype(spotting)::value) {
                                            hit[h] |= ok1 && q1 < lim32 ? 1u << j1 : 0u;
                                            hit[h] |= ok2 && q2 < lim32 ? 1u << j2 : 0u;
                                        }
                                    } else {
                                        least = fminf(least, fminf(q1, q2));
                                        pull(e1.w, dx1, dy1, dz1, q1, true);
                                        pull(e2.w, dx2, dy2, dz2, q2, both);
                                        if (decltype(spotting)::value) {
                                            hit[h] |= q1 < lim32 ? 1u << j1 : 0u;
                                            hit[h] |= q2 < lim32 ? 1u << j2 : 0u;
                                        }
                                    }
                                });
                            }
                        };
                        if (spot) sweep(std::integral_constant<bool, KIND == 1>{}, std::false_type{});
                        else sweep(std::false_type{}, std::false_type{});
                        if (__any(!(least > r2min) || cx != cx)) {
                            cx = cy = cz = 0.f;
                            if (spot) sweep(std::integral_constant<bool, KIND == 1>{}, std::true_type{});
                            else sweep(std::false_type{}, std::true_type{});
                        }
                    } else {
                        auto sweep = [&](auto spotting) {
                            for (int h = 0; h < kHalves; h++) {
                                auto one = [&](int j) {
                                    const float4 e = fs[32 * half0 + j];
                                    const float dx = e.x - xr, dy = e.y - yr, dz = e.z - zr;
                                    const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                                    pull(e.w, dx, dy, dz, r2, true);
                                    if (decltype(spotting)::value) hit[h] |= r2 < lim32 ? 1u << (j & 31) : 0u;
                                };
                                // the lane's field, or (TPG 64, uniform) this half of the chunk
                                int j = TPG == 64 ? 32 * h : TPG * sub - 32 * half0;
                                const int je = TPG == 64 ? (cnt < 32 * h + 32 ? cnt : 32 * h + 32)
                                                         : (cnt - 32 * half0 < j + TPG ? cnt - 32 * half0 : j + TPG);
                                for (; j + 4 <= je; j += 4) { one(j); one(j + 1); one(j + 2); one(j + 3); }
                                for (; j < je; j++) one(j);
                                // A lane takes all 64 entries here, where it
                                // meets a fifth of a partial chunk's: two
                                // plain sums of 32.  (rms error of an acceleration
                                // on the 1 M disk 8.7e-8 with one sum of 64, now
                                // 7.5e-8; four sums of 16 7.0e-8, but the walk
                                // 685 -> 702 us.)
                                if (TPG == 64 && h == 0) settle();
                            }
                        };
                        if (spot) sweep(std::integral_constant<bool, KIND == 1>{});
                        else sweep(std::false_type{});
                    }
                    const unsigned long long exz = __ballot(left != 0);   // lanes left out of some entry of this chunk
                    if (exz) {
                        // the left-out lanes, entry by entry (rare: close pairs, or
                        // a group whose box is far wider than its neighbours' gaps)
                        float elx = 0.f, ely = 0.f, elz = 0.f;
                        if (!dfc && lane < cnt) {
                            const core::TreeNode w = a.tree[enode[e0 + lane]];
                            const double exd = (w.cx - gcx) * invL, eyd = (w.cy - gcy) * invL, ezd = (w.cz - gcz) * invL;
                            elx = (float)(exd - (double)(float)exd);
                            ely = (float)(eyd - (double)(float)eyd);
                            elz = (float)(ezd - (double)(float)ezd);
                        }
                        for (int jj = 0; jj < cnt; jj++) {
                            const unsigned long long Mj = rl(emask, jj);
                            if (!(Mj & exz)) continue;
                            const float4 e = fs[jj];
                            float dx = e.x - xr, dy = e.y - yr, dz = e.z - zr;
                            float lx, ly, lz;
                            if (dfc) { const float4 l = fl[jj]; lx = l.x; ly = l.y; lz = l.z; }
                            else { lx = rl(elx, jj); ly = rl(ely, jj); lz = rl(elz, jj); }
                            unsigned long long Z1;
                            if (dfc) {
                                Z1 = Mj;   // every lane of the entry is tested again below
                            } else {
                                const float r2p = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                                Z1 = Mj & ~__ballot(r2p > r2min);
                            }
                            if (!Z1) continue;
                            dx += lx - xlo; dy += ly - ylo; dz += lz - zlo;
                            const float r2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
                            const unsigned long long Z = Z1 & ~__ballot(r2 > r2df);
                            if (!dfc) {
                                const unsigned long long okD = Z1 & ~Z;
                                if (okD) {
                                    pull(e.w, dx, dy, dz, r2, in_mask(okD));
                                    if (KIND == 1 && in_mask(okD & sphB & __ballot(r2 < lim32))) hb |= 1ull << jj;
                                }
                            }
                            if (Z) {
                                if (lane == 0 && nrec < kNearRecs) {
                                    a.near_node[(size_t)g * kNearRecs + nrec] = enode[e0 + jj];
                                    a.near_mask[(size_t)g * kNearRecs + nrec] = TPG == 64 ? Z : Z >> (TPG * (jj / TPG));
                                }
                                nrec++;
                                nint -= (unsigned long long)__builtin_popcountll(Z);
                                // as SPH candidates they go on the lists as they are
                                // (the pair kernel skips r == 0)
                                if (KIND == 1 && in_mask(Z & sphB)) hb |= 1ull << jj;
                            }
                        }
                        dfmode = true;   // the rest of this group's chunks carry the remainders
                    }
                    settle();
                } else {
                    const double4 *ds4 = S.e.d;
                    // the chunk's sums, added to the total after it: one plain
                    // sum over the thousand entries a target meets rounds three
                    // times as much (rms error on the 1 M disk 5.1e-16, so
                    // 1.9e-16, the time the same)
                    double cx = 0.0, cy = 0.0, cz = 0.0;
                    auto sweep = [&](auto spotting) {
                        for (int h = 0; h < kHalves; h++) {
                            auto one = [&](int j, bool on) {
                                const double4 e = ds4[32 * (half0 + h) + j];
                                const double dx = e.x - px, dy = e.y - py, dz = e.z - pz;
                                const double r2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
                                if (KIND == 4) {
                                    // -(G / e0) m (pi/2 - atan(r / e0)), scaled at the end
                                    // (neither 0 nor inf: where r^2 overflows nothing is
                                    // left of the pair, and it has no root)
                                    if (__builtin_amdgcn_class(r2, 0x183) && on) {
                                        const double ir = rsq_full(r2);
                                        s.pot = __builtin_fma(e.w, softened_angle(a.wp.e0, r2 * ir, ir), s.pot);
                                        lnint++;
                                    }
                                    return;
                                }
                                double gx, gy, gz;
                                const bool ok = on && r2 != 0.0 &&
                                                core::soft_force(e.w, dx, dy, dz, sqrt(r2), a.wp, &gx, &gy, &gz);
                                if (ok) { cx += gx; cy += gy; cz += gz; lnint++; }
                                if (decltype(spotting)::value) hit[h] |= ok && r2 < lim64 ? 1u << j : 0u;
                            };
                            if (KIND == 4 || a.wp.soft_live) {
                                bit_pairs(word[h], [&](int j1, int j2, bool both) { one(j1, true); one(j2, both); });
                                continue;
                            }
                            // Two entries side by side, with nothing between
                            // them but the rare case: f = m / ((r^2 + e^2) r) as
                            // one reciprocal root of r^2 (r^2 + e^2)^2.  (A root
                            // and a quotient took half as many instructions
                            // again: the 1 M disk's walk 1,192 us, now 1,000; one
                            // entry at a time, with the rare case between
                            // two, 1,236.)
                            auto two = [&](int j1, int j2, bool both) {
                                const double4 e1 = ds4[32 * (half0 + h) + j1], e2 = ds4[32 * (half0 + h) + j2];
                                double dx1 = e1.x - px, dy1 = e1.y - py, dz1 = e1.z - pz;
                                double dx2 = e2.x - px, dy2 = e2.y - py, dz2 = e2.z - pz;
                                const double q1 = __builtin_fma(dx1, dx1, __builtin_fma(dy1, dy1, dz1 * dz1));
                                const double q2 = __builtin_fma(dx2, dx2, __builtin_fma(dy2, dy2, dz2 * dz2));
                                const double s1 = q1 + e02, s2 = q2 + e02;
                                const double x1 = (q1 * s1) * s1, x2 = (q2 * s2) * s2;
                                double f1 = e1.w * rsq_full(x1), f2 = e2.w * rsq_full(x2);
                                bool ok1 = x1 > 0x1p-900 && fabs(f1) < 0x1p1000;
                                bool ok2 = x2 > 0x1p-900 && fabs(f2) < 0x1p1000;
                                if (__any(!(ok1 && ok2))) {
                                    // coincident, NaN, or far outside the scales
                                    // of a simulation: r2 == 0 gives NaN and is
                                    // skipped like any NaN
                                    auto rare = [&](double m, double r2, double &dx, double &dy, double &dz, double &f,
                                                    bool &ok) {
                                        if (ok) return;
                                        const double ri = rsq_full(r2), rr = r2 * ri;
                                        f = m * rcp_full(rr * rr + e02) * ri;
                                        ok = !__builtin_isunordered(f * dx, f * dy) && f * dz == f * dz;
                                        if (!ok) f = dx = dy = dz = 0.0;
                                    };
                                    rare(e1.w, q1, dx1, dy1, dz1, f1, ok1);
                                    rare(e2.w, q2, dx2, dy2, dz2, f2, ok2);
                                }
                                ok2 = ok2 && both;
                                f2 = both ? f2 : 0.0;
                                cx = __builtin_fma(f2, dx2, __builtin_fma(f1, dx1, cx));
                                cy = __builtin_fma(f2, dy2, __builtin_fma(f1, dy1, cy));
                                cz = __builtin_fma(f2, dz2, __builtin_fma(f1, dz1, cz));
                                lnint += (ok1 ? 1u : 0u) + (ok2 ? 1u : 0u);
                                if (decltype(spotting)::value) {
                                    hit[h] |= ok1 && q1 < lim64 ? 1u << j1 : 0u;
                                    hit[h] |= ok2 && q2 < lim64 ? 1u << j2 : 0u;
                                }
                            };
                            // (in groups of 64; with fewer targets the loop's
                            // registers spill)
                            if (TPG < 64 || part) {
                                bit_pairs(word[h], two);
                            } else if (mine) {
                                int j = 0;
                                const int je = cnt - 32 * h < 32 ? cnt - 32 * h : 32;
                                for (; j + 2 <= je; j += 2) two(j, j + 1, true);
                                if (j < je) two(j, j, false);
                            }
                        }
                    };
                    if (spot) sweep(std::integral_constant<bool, KIND == 1>{});
                    else sweep(std::false_type{});
                    s.ax += cx;
                    s.ay += cy;
                    s.az += cz;
                }
                // The candidates found go on their target's list in entry
                // order (TPG < 64: the NS lanes of a target one after another)
                if (spot) {
                    unsigned long long hm = hit[0];
                    if (kHalves == 2) hm |= (unsigned long long)hit[kHalves - 1] << 32;
                    else hm <<= 32 * half0;
                    hm = (hm | hb) & candB;
                    int at = lcnt, add = __builtin_popcountll(hm);
                    for (int d = TPG; d < 64; d <<= 1) {
                        const int o = __shfl_xor(add, d, 64);
                        if (lane & d) at += o;
                        add += o;
                    }
                    if (a.spill_cap == 0) {   // uniform
                        for (; hm; hm &= hm - 1, at++)
                            if (at < kSphK) lbase[at] = enode[e0 + __builtin_ctzll(hm)];
                        lcnt += add;
                    } else {
                        // a step adds at most 64, so it enters one new chunk at most
                        const int chunk = lcnt > 0 ? (lcnt - 1) / kSphK : 0;
                        lcnt += add;
                        int32_t *nbase = lbase;
                        const bool full = add > 0 && (lcnt - 1) / kSphK > chunk;
                        if (__any(full)) {
                            int c = -1;
                            if (full && sub == 0 && chunk < kSphMore && lbase) {
                                c = atomicAdd(&a.dsw->spill_next, 1);
                                if (c >= a.spill_cap) c = -1;
                                else a.sph_more[(size_t)slot * kSphMore + chunk] = c;
                            }
                            c = shfl_i(c, tl);
                            if (full) nbase = c >= 0 ? a.sph_spill + (size_t)c * kSphK : nullptr;
                        }
                        for (; hm; hm &= hm - 1, at++) {
                            int32_t *to = at / kSphK == chunk ? lbase : nbase;
                            if (to) to[at % kSphK] = enode[e0 + __builtin_ctzll(hm)];
                        }
                        lbase = nbase;
                    }
                }
                // SPH term.  Pairs (target lane t, entry j) with r < 2 h_t are
                // queued in LDS as they are found and evaluated 64 at a time,
                // one pair per lane: the lane loads t's state (key order) and
                // j's node record again rather than keeping them in
                // registers through the walk, and stages the pair's result in
                // LDS by its queue slot (the staging area, free once the
                // chunk's gravity loop is done).  Each target lane then adds
                // its own pairs' results in slot order, so the sums do not
                // depend on timing.
                if (KIND == 2 && sphB) {
                    if (candB) {
                        double *acc = &S.e.acc[0][0];
                        uint16_t *pairs = reinterpret_cast<uint16_t *>(S.ent_full);   // unused by this kind
                        int np = 0;
                        auto run_pairs = [&](int base, int cntp) {
                            wave_sync_lds();
                            const int pr = lane < cntp ? (int)pairs[base + lane] : 0;
                            const int jl = pr >> 8;
                            double wax = 0.0, way = 0.0, waz = 0.0, wdu = 0.0;
                            if (lane < cntp) {
                                const int tl = pr & 63;
                                const int ti = g * 64 + tl;
                                const double tx = a.sx[ti], ty = a.sy[ti], tz = a.sz[ti];
                                const double tvx = a.svx[ti], tvy = a.svy[ti], tvz = a.svz[ti];
                                core::Target tt;
                                tt.h = a.h[ti]; tt.rho = a.rho[ti]; tt.P = a.P[ti];
                                const core::SphNode nj = a.tsph[S.ent_node[e0 + jl]];   // (a candidate has gas)
                                const double jx = nj.cx, jy = nj.cy, jz = nj.cz, jg = nj.gas;
                                const double jvx = nj.vx, jvy = nj.vy, jvz = nj.vz;
                                const core::SphConst k = core::sph_const(tt);
                                core::WalkSums w{0, 0, 0, 0, 0, 0, 0};
                                const double ddx = tx - jx, ddy = ty - jy, ddz = tz - jz;
                                const double r2 = ddx * ddx + ddy * ddy + ddz * ddz;
                                sph_pair(ddx, ddy, ddz, r2, jg, tvx - jvx, tvy - jvy, tvz - jvz, k, &w);
                                wax = w.ax; way = w.ay; waz = w.az; wdu = w.du;
                                s.nsph += w.nsph;
                            }
                            acc[lane] = wax; acc[64 + lane] = way; acc[128 + lane] = waz; acc[192 + lane] = wdu;
                            wave_sync_lds();
                            for (int k = 0; k < cntp; k++) {
                                if (((int)pairs[base + k] & 63) == lane) {
                                    s.ax += acc[k]; s.ay += acc[64 + k]; s.az += acc[128 + k]; s.du += acc[192 + k];
                                }
                            }
                        };
                        for (unsigned long long cb = candB; cb; cb &= cb - 1) {
                            const int j = __builtin_ctzll(cb);
                            const unsigned long long W = rl(emask, j) & sphB;
                            if (!W) continue;
                            const double jx = rl(ecx, j), jy = rl(ecy, j), jz = rl(ecz, j);
                            bool inside = false;
                            if (in_mask(W)) {
                                const double ddx = px - jx, ddy = py - jy, ddz = pz - jz;
                                const double r2 = ddx * ddx + ddy * ddy + ddz * ddz;
                                if (r2 != 0.0) {
                                    if (r2 < h2x4 * (1.0 - 1e-12)) inside = true;
                                    else if (!(r2 > h2x4 * (1.0 + 1e-12))) inside = sqrt(r2) < a.h[q] * 2;
                                }
                            }
                            const unsigned long long I = __ballot(inside);
                            if (inside) pairs[np + mbcnt(I)] = (uint16_t)(lane | (j << 8));
                            np += __builtin_popcountll(I);
                            if (np >= 64) {
                                run_pairs(np - 64, 64);
                                np -= 64;
                            }
                        }
                        if (np > 0) run_pairs(0, np);
                    }
                }
                n_entries += (unsigned long long)cnt;
                if (part) ni -= cnt; else nf -= cnt;
            }
            if (sp == 0 && ni + nf == 0) break;
        }
        if (KIND != 2 && KIND != 4 && lane == 0) {
            bin_add(a.cbins, kCntEntries, g, n_entries);
            bin_add(a.cbins, kCntTests, g, n_tests);
            bin_add(a.cbins, kCntMixed, g, n_mixed);
        }
    }
    if (KIND == 2) {
        // SPH of overflowed targets, added to their gravity
        if (sph_lane) {
            a.ax[q] += s.ax; a.ay[q] += s.ay; a.az[q] += s.az;
            a.dUdt[q] += s.du;
        }
        unsigned long long cs = wave_sum_u64((unsigned long long)s.nsph);
        if (lane == 0) bin_add(a.cbins, kCntSphPairs, g, cs);
        return;
    }
    if (KIND == 4) {
        double ph = s.pot;
        int any = lnint != 0u;
        for (int d = TPG; d < 64; d <<= 1) {
            ph += __shfl_xor(ph, d, 64);
            any |= __shfl_xor(any, d, 64);
        }
        if (valid_t && sub == 0) a.pot[q] = any ? -(a.wp.G / a.wp.e0) * ph : 0.0;
        return;
    }
    double ox, oy, oz;
    if (F32) {
        // (a full chunk's sweep knows no mask: lanes whose target takes no part,
        // a massless one among them, have summed what was not theirs)
        const double scale = a.nn > 0 ? a.wp.G * a.tree[0].mass * invL * invL : 0.0;
        ox = mine ? (double)sumx * scale : 0.0;
        oy = mine ? (double)sumy * scale : 0.0;
        oz = mine ? (double)sumz * scale : 0.0;
    } else {
        ox = s.ax; oy = s.ay; oz = s.az;
    }
    // the NS lanes of a target in a fixed order
    for (int d = TPG; d < 64; d <<= 1) {
        ox += __shfl_xor(ox, d, 64);
        oy += __shfl_xor(oy, d, 64);
        oz += __shfl_xor(oz, d, 64);
    }
    if (act && sub == 0) { a.ax[q] = ox; a.ay[q] = oy; a.az[q] = oz; }
    if (KIND == 1 && slot >= 0 && sub == 0) {
        a.sph_cnt[slot] = lcnt;
        if (lcnt > kSphK) a.gover[t >> 6] = 1;
    }
    if (KIND == 1) {
        // targets whose candidates did not fit their list alone
        const unsigned long long ovB = __ballot(slot >= 0 && sub == 0 && lcnt > kSphK);
        if (lane == 0) bin_add(a.cbins, kCntSphOver, g, (unsigned long long)__builtin_popcountll(ovB));
    }
    nint += wave_sum_u64((unsigned long long)lnint);
    if (F32) {
        if (lane == 0) a.near_cnt[g] = nrec;
        // a group walked again in FP64 (KIND 3) counts its interactions there
        if (nrec > kNearRecs) nint = 0ull;
    }
    if (lane == 0) bin_add(a.cbins, kCntInteractions, g, nint);
}

__device__ inline int wave_group() {
    return walk_workgroup(blockIdx.x, gridDim.x) * kWaves + (int)(threadIdx.x >> 6);
}

// Targets per walk group for a set of n particles.  A group is one wave, and
// the walk of a small set is one wave's latency: with 64 targets per group a
// set of 10,000 has 157 waves for the chip's 1,024 SIMDs.  Groups of 8 or 16
// targets give eight or four times the waves, each with a smaller box (fewer
// nodes) and its sweep split over the 64 / TPG lanes of a target; the whole
// walk does more traversal work (2.1 and 1.3 times the node tests per lane of
// a SIMD), which costs once the SIMDs have waves to overlap: groups of 8 up to
// the 4,096 waves the chip holds at once.  Walk kernel, microseconds, groups
// of 8 / 16 / 64: Plummer 10,000 FP32 39 / 51 / 130; 24,576 FP32 54 / 64 / -;
// 32,768 FP32 57 / 62 / -, FP64 60 / 68 / -; 33,333 FP64 69 / 69 / -; disk
// 28,000 FP32 67 / 79 / -; 32,768 FP32 75 / 84 / -, FP64 76 / 86 / -; 100,000
// FP64 - / 167 / 254; 150,000 FP32 - / 181 / 224; 200,000 FP32 - / 231 / 246,
// FP64 - / 273 / 307; 400,000 FP64 - / 495 / 503; 450,000 FP64 - / 552 / 542;
// 1 M FP32 - / 1014 / 690, FP64 - / 1147 / 1000.  In FP32 the two draw level
// above: 250,000 disk 265 / 295, Hernquist 226 / 246, Plummer 216 / 206 (at
// opening angle 0.15 2,610 / 3,325, 2,500 / 3,085, 2,295 / 2,545); 275,000 291 /
// 269, 242 / 242, 238 / 254; 400,000 393 / 391, 325 / 329, 322 / 310.  The
// choice depends on the set alone, so a job of a batched walk has the
// arithmetic of a walk of its own.
constexpr int kTpg8Max = 32768, kTpg16Max32 = 262144, kTpg16Max64 = 400000;
inline int walk_tpg(int64_t n, bool f32) {
    return n <= kTpg8Max ? 8 : n <= (f32 ? kTpg16Max32 : kTpg16Max64) ? 16 : 64;
}

// Kernels per precision form: gravity with SPH candidate recording (any gas
// uploaded) or plain gravity, and the overflow SPH walk (FP64 for both forms).
#define AG2_WALK_BOUNDS __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))

__global__ AG2_WALK_BOUNDS void k_walk_block64(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<false, 1, 64>(a, wave_group(), lds);
}

__global__ AG2_WALK_BOUNDS void k_walk_block64_nogas(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<false, 0, 64>(a, wave_group(), lds);
}

__global__ AG2_WALK_BOUNDS void k_walk_block32(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<true, 1, 64>(a, wave_group(), lds);
}

__global__ AG2_WALK_BOUNDS void k_walk_block32_nogas(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<true, 0, 64>(a, wave_group(), lds);
}

// ... in groups of fewer targets (walk_tpg)
template <bool F32, int KIND, int TPG>
__global__ AG2_WALK_BOUNDS void k_walk_small(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<F32, KIND, TPG>(a, wave_group(), lds);
}

// The potential (energy diagnostics): the same walk, the softened potential
// in place of the force.  One lane per target walking the pre-order nodes by
// itself took 3.58 ms on the 1 M disk (uncoalesced records, a square root, a
// quotient and the library's atan per pair); this takes 1.20 ms.
template <int TPG>
__global__ AG2_WALK_BOUNDS void k_walk_potential(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<false, 4, TPG>(a, wave_group(), lds);
}

// The overflow walk and the near pass usually touch few groups, but a
// small opening angle can flag thousands (every SPH list overflowing, many
// near pairs): one wave per group, exiting at once when its group is not
// flagged, keeps those walks in parallel.
__global__ AG2_WALK_BOUNDS void k_walk_sph_overflow(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    walk_block<false, 2, 64>(a, wave_group(), lds);   // exits unless the group is flagged in gover
}

// The near pairs of a split-precision walk in FP64 on the FP64 positions,
// the reference's law (Node.cpp:337-365; r == 0 skipped, Node.cpp:274-276),
// added to the walk's results in record order.  Groups with more records
// than kept are walked again in FP64 instead (k_near_pass).
template <int TPG>
__device__ inline void near_fp64_group(const WalkArgs &a, int g, int cnt) {
    const int lane = lane_id();
    const int t = g * TPG + lane;   // lanes past TPG are in no record's mask
    double px = 0.0, py = 0.0, pz = 0.0;
    if (t < a.n) { px = a.sx[t]; py = a.sy[t]; pz = a.sz[t]; }
    double fx = 0.0, fy = 0.0, fz = 0.0;
    unsigned long long nint = 0ull, any = 0ull, npairs = 0ull;
    for (int k = 0; k < cnt; k++) {
        const int node = a.near_node[(size_t)g * kNearRecs + k];
        const unsigned long long M = a.near_mask[(size_t)g * kNearRecs + k];
        any |= M;
        npairs += (unsigned long long)__builtin_popcountll(M);
        bool live = false;
        if (in_mask(M)) {
            const core::TreeNode w = a.tree[node];
            const double dx = w.cx - px, dy = w.cy - py, dz = w.cz - pz;
            const double r2 = dx * dx + dy * dy + dz * dz;
            if (r2 != 0.0) {
                live = true;
                const double r = sqrt(r2);
                const double f = a.wp.G * w.mass / (r * r + a.wp.e0 * a.wp.e0);
                fx += f * (dx / r); fy += f * (dy / r); fz += f * (dz / r);
            }
        }
        nint += (unsigned long long)__builtin_popcountll(__ballot(live));
    }
    if (in_mask(any)) { a.ax[t] += fx; a.ay[t] += fy; a.az[t] += fz; }
    if (lane == 0) {
        bin_add(a.cbins, kCntInteractions, g, nint);
        bin_add(a.cbins, kCntNear, g, npairs);
    }
}

// The near pass: groups with at most kNearRecs recorded pairs evaluate them
// in FP64 (near_fp64_group); groups with more are walked again in FP64.
template <int TPG>
__global__ AG2_WALK_BOUNDS void k_near_pass(WalkArgs a) {
    __shared__ BlockLds lds[kWaves];
    const int g = wave_group();
    if (g >= (a.n + TPG - 1) / TPG) return;
    const int cnt = a.near_cnt[g];
    if (cnt > kNearRecs) {
        if (lane_id() == 0) bin_add(a.cbins, kCntNearRedo, g, 1ull);
        walk_block<false, 3, TPG>(a, g, lds);
    } else if (cnt > 0) {
        near_fp64_group<TPG>(a, g, cnt);
    }
}

// Batched walk of several independent simulations (a serving round): job j
// owns the global groups [group0[j], group0[j + 1]); a wave finds its job by
// binary search and walks that job's tree for its own targets, so each job's
// arithmetic is the same as in a walk of its own.
struct JobWalk {
    WalkArgs a;
    int group0;
    int tpg;   // targets per group (walk_tpg of the job's own n)
};

__device__ inline int find_job(const JobWalk *jobs, int nj, int G) {
    int lo = 0, hi = nj - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].group0 <= G) lo = mid; else hi = mid - 1;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

template <bool F32, int KIND>
__device__ __forceinline__ void walk_jobs(const JobWalk *jobs, int nj, int total, BlockLds *lds) {
    const int G = wave_group();
    if (G >= total) return;   // whole waves only: nothing below synchronises across waves
    const int j = find_job(jobs, nj, G);
    const int g = G - jobs[j].group0, tpg = jobs[j].tpg;
    if (tpg == 64) walk_block<F32, KIND, 64>(jobs[j].a, g, lds);
    else if (tpg == 16) walk_block<F32, KIND, 16>(jobs[j].a, g, lds);
    else walk_block<F32, KIND, 8>(jobs[j].a, g, lds);
}

__global__ AG2_WALK_BOUNDS void k_walk_jobs64(const JobWalk *jobs, int nj, int total) {
    __shared__ BlockLds lds[kWaves];
    walk_jobs<false, 1>(jobs, nj, total, lds);
}
__global__ AG2_WALK_BOUNDS void k_walk_jobs64_nogas(const JobWalk *jobs, int nj, int total) {
    __shared__ BlockLds lds[kWaves];
    walk_jobs<false, 0>(jobs, nj, total, lds);
}
__global__ AG2_WALK_BOUNDS void k_walk_jobs32(const JobWalk *jobs, int nj, int total) {
    __shared__ BlockLds lds[kWaves];
    walk_jobs<true, 1>(jobs, nj, total, lds);
}
__global__ AG2_WALK_BOUNDS void k_walk_jobs32_nogas(const JobWalk *jobs, int nj, int total) {
    __shared__ BlockLds lds[kWaves];
    walk_jobs<true, 0>(jobs, nj, total, lds);
}


// Active SPH targets (gas, h > 0, due this step) in key order get list
// slots: per-tile counts, a one-workgroup scan, the scatter.  The count
// pass also clears gslot and the groups' overflow flags.
__global__ __launch_bounds__(256) void k_sph_count(int n, const uint8_t *type, const double *h,
                                                   const uint8_t *active, const double *m, int32_t *tiles,
                                                   int32_t *gslot, uint8_t *gover, DevState *ds) {
    __shared__ int scr[4];
    if (blockIdx.x == 0 && threadIdx.x == 0) ds->spill_next = 0;
    int b0 = blockIdx.x * 1024 + threadIdx.x * 4;
    int c = 0;
    for (int k = 0; k < 4; k++) {
        int i = b0 + k;
        if (i < n) {
            gslot[i] = -1;
            if ((i & 63) == 0) gover[i >> 6] = 0;
            c += (type[i] == 2 && h[i] > 0.0 && active[i] && m[i] != 0.0) ? 1 : 0;
        }
    }
    int tot;
    block256_excl_scan(c, scr, &tot);
    if (threadIdx.x == 0) tiles[blockIdx.x] = tot;
}

// The active SPH targets in key order: each tile forms its offset from the
// tile counts; tile 0 records their number.
__global__ __launch_bounds__(256) void k_sph_scatter(int n, const uint8_t *type, const double *h,
                                                     const uint8_t *active, const double *m,
                                                     const int32_t *tiles, int32_t *gidx, int32_t *gslot,
                                                     DevState *ds) {
    __shared__ int scr[4];
    int b0 = blockIdx.x * 1024 + threadIdx.x * 4;
    int f[4], c = 0;
    for (int k = 0; k < 4; k++) {
        int i = b0 + k;
        f[k] = (i < n && type[i] == 2 && h[i] > 0.0 && active[i] && m[i] != 0.0) ? 1 : 0;
        c += f[k];
    }
    int tot;
    const int pre = tile_offset(tiles, (int)gridDim.x, (int)blockIdx.x, scr, &tot);
    if (blockIdx.x == 0 && threadIdx.x == 0) ds->n_sph = tot;
    int off = block256_excl_scan(c, scr, nullptr) + pre;
    for (int k = 0; k < 4; k++)
        if (f[k]) { gidx[off] = b0 + k; gslot[b0 + k] = off; off++; }
}

// The SPH term (Node::calcSPHForce, Node.cpp:88-172) of every recorded
// (target, node) candidate.  Eight lanes per target stride through its
// list; the four sums are then reduced over the eight lanes in a fixed
// butterfly order.  A candidate counts when r < 2 h (decided like the
// reference: on r^2 with a margin, exactly inside it), r != 0 and the node is
// not the target's own leaf.  Lists that overflowed are left to the overflow
// walk.
//
// Four neighbouring lanes read one record together, 16 bytes each, and hand
// the pieces to their owners through LDS: a lane that reads its own 64-byte
// record alone makes every load of the wave touch 64 cache lines, and the
// L1's tag lookups (256 cycles per 64 records) bounded the kernel.  With that
// and the short root and quotients (sph_pair_plain) 14.1 M pairs of the 1 M
// disk take 117 us where they took 136, 200,000 disk at opening angle 0.15
// 196 us for 224; the shared reads alone 124 and 212.  What is left is the
// vector unit (about half of the time), and four waves per SIMD to wait with:
// holding the registers to five or six spills (325 and 541 us).
constexpr int kPairLanes = 8;
constexpr int kQuadBytes = 4 * 64 + 64;   // records of a quad's four lanes, and room to spread the banks

// Piece j (16 bytes) of the record of lane i of quad q: the pieces of a
// record are permuted by i, so that eight lanes reading the same piece of
// their records meet no bank twice.
__device__ inline int piece_at(int q, int i, int j) { return q * kQuadBytes + i * 64 + (j ^ i) * 16; }

template <int I>
__device__ inline int quad_bcast(int v) {
    return __builtin_amdgcn_mov_dpp(v, I * 0x55, 0xf, 0xf, true);
}

// SPILL: lists may go on in spill chunks (the context has some).
template <bool SPILL>
__global__ __launch_bounds__(256) void k_sph_pairs(WalkArgs a, const int32_t *gidx, const int32_t *cnts) {
    static_assert(sizeof(core::SphNode) == 64, "a record is four pieces of 16 bytes");
    __shared__ __align__(16) char stage[4][16 * kQuadBytes];
    const int lane = lane_id();
    const int sub = lane & (kPairLanes - 1);
    char *mine = stage[threadIdx.x >> 6];
    const int qd = lane >> 2, qi = lane & 3;
    // targets in key order, in XCD ranges: neighbouring targets share most
    // of their candidate records, which then come from one L2
    const int slot = (int)((xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x) / kPairLanes);
    const int nsph = a.ds->n_sph;
    core::WalkSums s{0, 0, 0, 0, 0, 0, 0};
    int t = -1, c = 0;
    if (slot < nsph) {
        c = cnts[slot];
        if (!list_overflowed(a, c)) t = gidx[slot];
        else c = 0;
    }
    core::Target tg{};
    double vx = 0.0, vy = 0.0, vz = 0.0;
    core::SphConst sk{};
    double ih = 0.0, h2 = 0.0;
    bool plain = false;
    unsigned np = 0u;   // pairs counted on the short path
    if (t >= 0) {
        tg.x = a.sx[t]; tg.y = a.sy[t]; tg.z = a.sz[t];
        tg.h = a.h[t]; tg.rho = a.rho[t]; tg.P = a.P[t];
        vx = a.svx[t]; vy = a.svy[t]; vz = a.svz[t];
        sk = core::sph_const(tg);
        ih = 1.0 / tg.h;
        plain = plain_support(tg.h);
        h2 = tg.h * 2;
    }
    // candidate k of the list: kSphK in the list itself, then spill chunks
    const int32_t *lst = a.sph_list + (size_t)slot * kSphK;
    auto candidate = [&](int k) -> int {
        if (k >= c) return 0;   // (a record of no use; record 0 is there)
        if (SPILL && k >= kSphK)
            return a.sph_spill[(size_t)a.sph_more[(size_t)slot * kSphMore + k / kSphK - 1] * kSphK + k % kSphK];
        return lst[k];
    };
    int most = c;
    for (int d = 32; d >= kPairLanes; d >>= 1) {
        const int o = __shfl_xor(most, d, 64);
        most = o > most ? o : most;
    }
    most = __builtin_amdgcn_readfirstlane(most);
    // piece qi of the quad's four records, one round ahead; the list entry
    // two rounds ahead
    uint4 p0{}, p1{}, p2{}, p3{};
    auto fetch = [&](int rec) {
        const char *base = (const char *)a.tsph + 16 * qi;
        p0 = *(const uint4 *)(base + (size_t)quad_bcast<0>(rec) * 64);
        p1 = *(const uint4 *)(base + (size_t)quad_bcast<1>(rec) * 64);
        p2 = *(const uint4 *)(base + (size_t)quad_bcast<2>(rec) * 64);
        p3 = *(const uint4 *)(base + (size_t)quad_bcast<3>(rec) * 64);
    };
    int next = 0;
    if (most > 0) {
        fetch(candidate(sub));
        next = candidate(sub + kPairLanes);
    }
    for (int k0 = 0; k0 < most; k0 += kPairLanes) {
        *(uint4 *)(mine + piece_at(qd, 0, qi)) = p0;
        *(uint4 *)(mine + piece_at(qd, 1, qi)) = p1;
        *(uint4 *)(mine + piece_at(qd, 2, qi)) = p2;
        *(uint4 *)(mine + piece_at(qd, 3, qi)) = p3;
        wave_sync_lds();
        if (k0 + kPairLanes < most) {
            fetch(next);
            next = candidate(k0 + 2 * kPairLanes + sub);
        }
        const double2 cxy = *(const double2 *)(mine + piece_at(qd, qi, 0));
        const double2 czg = *(const double2 *)(mine + piece_at(qd, qi, 1));
        const double2 vxy = *(const double2 *)(mine + piece_at(qd, qi, 2));
        const double2 vzp = *(const double2 *)(mine + piece_at(qd, qi, 3));
        wave_sync_lds();
        const int pidx = (int)(unsigned)__builtin_bit_cast(unsigned long long, vzp.y);
        const double dx = tg.x - cxy.x, dy = tg.y - cxy.y, dz = tg.z - czg.x;
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double ux = vx - vxy.x, uy = vy - vxy.y, uz = vz - vzp.x;
        const double vd = ux * dx + uy * dy + uz * dz, hv = tg.h * vd;
        const bool cand = k0 + sub < c && pidx != t;
        const bool fast = plain && plain_pair(r2, vd, hv);
        if (cand && fast) {
            double ir;
            const double r = root_plain(r2, &ir);
            if (r < h2) {   // the reference's test itself
                sph_pair_plain(dx, dy, dz, r, ir, czg.y, ux, uy, uz, vd, hv, sk, ih, &s.ax, &s.ay, &s.az, &s.du);
                np++;
            }
        }
        if (__any(cand && !fast)) {
            if (cand && !fast && r2 != 0.0 && sqrt(r2) < sk.h * 2) sph_pair(dx, dy, dz, r2, czg.y, ux, uy, uz, sk, &s);
        }
    }
    for (int d = kPairLanes / 2; d >= 1; d >>= 1) {
        s.ax += __shfl_xor(s.ax, d, 64);
        s.ay += __shfl_xor(s.ay, d, 64);
        s.az += __shfl_xor(s.az, d, 64);
        s.du += __shfl_xor(s.du, d, 64);
    }
    if (t >= 0 && sub == 0) {
        a.ax[t] += s.ax; a.ay[t] += s.ay; a.az[t] += s.az;
        a.dUdt[t] += s.du;
    }
    unsigned long long cs = wave_sum_u64((unsigned long long)s.nsph + np);
    if (lane == 0) bin_add(a.cbins, kCntSphPairs, (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), cs);
}

__global__ __launch_bounds__(256) void k_fold_counters(unsigned long long *bins, DevState *ds) {
    fold_counter_bins(bins, ds);
}

__global__ void k_zero_job_counters(const JobWalk *jobs, int nj) {
    int j = blockIdx.x * 64 + threadIdx.x;
    if (j >= nj) return;
    DevState *ds = jobs[j].a.dsw;
    ds->interactions = 0ull;
    ds->sph_pairs = 0ull;
    ds->walk_entries = 0ull;
    ds->walk_tests = 0ull;
    ds->walk_mixed = 0ull;
    ds->sph_overflow = 0ull;
    ds->near_pairs = 0ull;
    ds->near_redo = 0ull;
}

// Spill chunks for n_gas targets at this opening angle.  Within 2h a target
// meets about 75 gas nodes at theta 0.5, 570 at 0.15 (the 200,000 disk), and
// their number grows as theta^-1.75 up to the particles themselves; half as
// many again are provided, over three quarters of the list (so from theta
// 0.37 down: noting the chunks costs the walk 3 % where no list needs them).
// At theta 0.15 the overflow walk of the lists that did not fit took 5.26 ms
// of a force evaluation of 9.1 ms; with the chunks it has nothing to do, and
// the evaluation takes 3.9 ms.
int64_t sph_spill_chunks(int64_t n_gas, double theta) {
    const double t = theta > 0.05 ? theta : 0.05;
    double per = 1.5 * 75.0 * pow(0.5 / t, 1.75) / kSphK - 0.75;
    if (!(per > 0.0) || n_gas <= 0) return 0;
    if (per > kSphMore) per = kSphMore;
    const double want = per * (double)n_gas + 64.0;
    return want < 0x7fffffff ? (int64_t)want : 0x7fffffff;
}

// The chunks a context's targets may take: those of its own gas and opening
// angle, however many more a context sized for larger sets holds (which lists
// run past them, and so the rounding of the SPH sums, is then a matter of the
// set alone), or none where it holds fewer.
int64_t spill_usable(const Ctx &c) {
    const int64_t own = sph_spill_chunks(c.gas_count, c.p.theta);
    return c.spill_cap >= own ? own : 0;
}

WalkArgs walk_args(Ctx &c) {
    WalkArgs a;
    a.n = (int)c.n; a.nin = c.nin; a.nn = c.n_nodes;
    a.tree = c.tnode;
    a.tsph = c.tsph;
    a.gslot = c.gslot; a.sph_list = c.sph_list; a.sph_cnt = c.sph_cnt; a.gover = c.gover;
    a.sph_spill = c.sph_spill; a.sph_more = c.sph_more; a.spill_cap = (int)spill_usable(c);
    a.sx = c.x; a.sy = c.y; a.sz = c.z; a.sm = c.m; a.stype = c.type;
    a.svx = c.vx; a.svy = c.vy; a.svz = c.vz;
    a.h = c.h; a.rho = c.rho; a.P = c.P; a.active = c.active;
    a.ds = c.ds;
    a.wp = core::WalkParams{c.p.theta, c.p.e0, c.p.G, core::soft_branch_live(c.p.e0)};
    a.ax = c.ax; a.ay = c.ay; a.az = c.az; a.dUdt = c.dUdt; a.pot = c.pot;
    a.dsw = c.ds;
    a.cbins = c.cbins;
    a.near_cnt = c.near_cnt; a.near_node = c.near_node; a.near_mask = c.near_mask;
    return a;
}

}  // namespace

size_t job_walk_bytes() { return sizeof(JobWalk); }

void forces_batch(Ctx *const *cs, int nc, hipStream_t st, int f32, void *scratch_dev, void *scratch_host) {
    if (nc <= 0) return;
    JobWalk *hj = (JobWalk *)scratch_host;
    bool gas = false;
    int total = 0;
    for (int k = 0; k < nc; k++) {
        hj[k].a = walk_args(*cs[k]);
        hj[k].group0 = total;
        hj[k].tpg = walk_tpg(cs[k]->n, f32 != 0);
        total += (int)((cs[k]->n + hj[k].tpg - 1) / hj[k].tpg);
        gas = gas || cs[k]->sph_active;
    }
    JobWalk *dj = (JobWalk *)scratch_dev;
    AG2_HIP(hipMemcpyAsync(dj, hj, sizeof(JobWalk) * (size_t)nc, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_zero_job_counters, dim3((nc + 63) / 64), dim3(64), 0, st, dj, nc);
    dim3 grid((total + kWaves - 1) / kWaves), block(64 * kWaves);
    if (f32) {
        if (gas) hipLaunchKernelGGL(k_walk_jobs32, grid, block, 0, st, dj, nc, total);
        else hipLaunchKernelGGL(k_walk_jobs32_nogas, grid, block, 0, st, dj, nc, total);
    } else {
        if (gas) hipLaunchKernelGGL(k_walk_jobs64, grid, block, 0, st, dj, nc, total);
        else hipLaunchKernelGGL(k_walk_jobs64_nogas, grid, block, 0, st, dj, nc, total);
    }
    AG2_HIP(hipGetLastError());
}

void fold_counters(Ctx &c) {
    static_assert(kCountBins == 256, "k_fold_counters runs one thread per bin");
    hipLaunchKernelGGL(k_fold_counters, dim3(1), dim3(256), 0, c.stream, c.cbins, c.ds);
    AG2_HIP(hipGetLastError());
}

int64_t sph_spill_bytes(int64_t n_gas, double theta) {
    const int64_t chunks = sph_spill_chunks(n_gas, theta);
    return chunks > 0 ? chunks * kSphK * 4 + n_gas * kSphMore * 4 : 0;
}

// Where there is no memory for the chunks the overflow walk does their work:
// past the share a pool allows, or half of what is free on the device (later
// buffers of the context, and other contexts, need theirs).
void reserve_spill(Ctx &c) {
    const int64_t want = sph_spill_chunks(c.sph_cap, c.p.theta);
    if (!c.sph_active || c.spill_cap >= want || c.spill_refused == want) return;
    const int64_t bytes = sph_spill_bytes(c.sph_cap, c.p.theta);
    if (c.spill_room >= 0 && bytes > c.spill_room) return;
    AG2_HIP(hipStreamSynchronize(c.stream));
    if (c.sph_spill) { (void)hipFree(c.sph_spill); c.sph_spill = nullptr; }
    if (c.sph_more) { (void)hipFree(c.sph_more); c.sph_more = nullptr; }
    c.spill_cap = 0;
    size_t avail = 0, all = 0;
    AG2_HIP(hipMemGetInfo(&avail, &all));
    if ((size_t)bytes > avail / 2 || hipMalloc(&c.sph_spill, (size_t)want * kSphK * 4) != hipSuccess ||
        hipMalloc(&c.sph_more, (size_t)c.sph_cap * kSphMore * 4) != hipSuccess) {
        (void)hipGetLastError();
        if (c.sph_spill) { (void)hipFree(c.sph_spill); c.sph_spill = nullptr; }
        c.sph_more = nullptr;
        c.spill_refused = want;
        return;
    }
    c.spill_cap = want;
}

// SPH candidate lists for a step: slots for the active SPH targets (before
// the gravity walk, which fills the lists) ...
void sph_prepare(Ctx &c) {
    if (!c.sph_active) return;
    reserve_spill(c);   // (a smaller theta than at the upload)
    hipStream_t st = c.stream;
    int n = (int)c.n;
    int nt = (n + 1023) / 1024;
    hipLaunchKernelGGL(k_sph_count, dim3(nt), dim3(256), 0, st, n, c.type, c.h, c.active, c.m, c.gtiles, c.gslot,
                       c.gover, c.ds);
    hipLaunchKernelGGL(k_sph_scatter, dim3(nt), dim3(256), 0, st, n, c.type, c.h, c.active, c.m, c.gtiles, c.gidx,
                       c.gslot, c.ds);
    AG2_HIP(hipGetLastError());
}

// ... and their evaluation after it, with the overflow walk for lists that
// did not fit (it exits at once for groups without one).
void sph_finish(Ctx &c) {
    if (!c.sph_active) return;
    hipStream_t st = c.stream;
    WalkArgs a = walk_args(c);
    int64_t lanes = c.gas_count * kPairLanes;
    int nb = (int)((lanes + 255) / 256);
    if (nb > 0 && a.spill_cap > 0) hipLaunchKernelGGL(k_sph_pairs<true>, dim3(nb), dim3(256), 0, st, a, c.gidx, c.sph_cnt);
    else if (nb > 0) hipLaunchKernelGGL(k_sph_pairs<false>, dim3(nb), dim3(256), 0, st, a, c.gidx, c.sph_cnt);
    const int groups = (int)((c.n + 63) / 64);
    hipLaunchKernelGGL(k_walk_sph_overflow, dim3((groups + kWaves - 1) / kWaves), dim3(64 * kWaves), 0, st, a);
    AG2_HIP(hipGetLastError());
}

// After a split-precision walk: the near pairs in FP64, then the groups with
// too many of them walked again in FP64 (both exit at once for other groups).
void near_finish(Ctx &c) {
    WalkArgs a = walk_args(c);
    const int tpg = walk_tpg(c.n, true);
    const int groups = (int)((c.n + tpg - 1) / tpg);
    const dim3 grid((groups + kWaves - 1) / kWaves), block(64 * kWaves);
    if (tpg == 64) hipLaunchKernelGGL(k_near_pass<64>, grid, block, 0, c.stream, a);
    else if (tpg == 16) hipLaunchKernelGGL(k_near_pass<16>, grid, block, 0, c.stream, a);
    else hipLaunchKernelGGL(k_near_pass<8>, grid, block, 0, c.stream, a);
    AG2_HIP(hipGetLastError());
}

int64_t walk_groups_max(int64_t cap) {
    int64_t most = cap / 64;
    const int64_t at[2][2] = {{kTpg8Max, 8}, {kTpg16Max32, 16}};   // the records are the split form's
    for (const auto &r : at) {
        const int64_t g = (cap < r[0] ? cap : r[0]) / r[1];
        most = g > most ? g : most;
    }
    return most + 1;
}

// The gravity walk of one context, in groups of walk_tpg targets.
template <bool F32>
static void launch_walk(Ctx &c) {
    const WalkArgs a = walk_args(c);
    const int tpg = walk_tpg(c.n, F32);
    const int groups = (int)((c.n + tpg - 1) / tpg);
    const dim3 grid((groups + kWaves - 1) / kWaves), block(64 * kWaves);
    hipStream_t st = c.stream;
    const bool gas = c.sph_active;
    if (tpg == 8) {
        if (gas) hipLaunchKernelGGL((k_walk_small<F32, 1, 8>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((k_walk_small<F32, 0, 8>), grid, block, 0, st, a);
    } else if (tpg == 16) {
        if (gas) hipLaunchKernelGGL((k_walk_small<F32, 1, 16>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((k_walk_small<F32, 0, 16>), grid, block, 0, st, a);
    } else if (F32) {
        if (gas) hipLaunchKernelGGL(k_walk_block32, grid, block, 0, st, a);
        else hipLaunchKernelGGL(k_walk_block32_nogas, grid, block, 0, st, a);
    } else {
        if (gas) hipLaunchKernelGGL(k_walk_block64, grid, block, 0, st, a);
        else hipLaunchKernelGGL(k_walk_block64_nogas, grid, block, 0, st, a);
    }
}

void forces(Ctx &c, int mode, bool fold) {
    hipStream_t st = c.stream;
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[4], st));
    if (mode == 0) {
        sph_prepare(c);
        if (c.timing >= 1) AG2_HIP(hipEventRecord(c.ev[8], st));
        launch_walk<false>(c);
        if (c.timing >= 1) AG2_HIP(hipEventRecord(c.ev[9], st));
        sph_finish(c);
        if (fold) fold_counters(c);
    } else {
        const WalkArgs a = walk_args(c);
        const int tpg = walk_tpg(c.n, false);
        const int groups = (int)((c.n + tpg - 1) / tpg);
        const dim3 grid((groups + kWaves - 1) / kWaves), block(64 * kWaves);
        if (tpg == 8) hipLaunchKernelGGL(k_walk_potential<8>, grid, block, 0, st, a);
        else if (tpg == 16) hipLaunchKernelGGL(k_walk_potential<16>, grid, block, 0, st, a);
        else hipLaunchKernelGGL(k_walk_potential<64>, grid, block, 0, st, a);
    }
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[5], st));
    AG2_HIP(hipGetLastError());
}

// The split-precision sweep works in units of the root half-width R, and its
// force m' / sqrt(r'^2 (r'^2 + e'^2)^2) needs (e0 / R)^4 well inside the FP32
// exponent range.  When R has grown far beyond the softening length (escaped
// particles can push it to 1e24 kpc), the FP64 sweep runs instead.
bool fp32_usable(const Ctx &c) {
    const double R = __builtin_bit_cast(double, c.hs.Rbits);
    return !(R > 0.0) || c.p.e0 >= ldexp(R, -24);
}

void forces_fp32(Ctx &c, int mode, bool fold) {
    if (mode != 0) return forces(c, mode);
    hipStream_t st = c.stream;
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[4], st));
    sph_prepare(c);
    if (c.timing >= 1) AG2_HIP(hipEventRecord(c.ev[8], st));
    launch_walk<true>(c);
    if (c.timing >= 1) AG2_HIP(hipEventRecord(c.ev[9], st));
    near_finish(c);
    sph_finish(c);
    if (fold) fold_counters(c);
    if (c.timing >= 2) AG2_HIP(hipEventRecord(c.ev[5], st));
    AG2_HIP(hipGetLastError());
}

}  // namespace ag2
