// knn.hip -- k-nearest-neighbor and radius search over the column grid, fused
// with the neighborhood covariance; plus the per-row eigensolve and
// stage-output kernel.
//
// Replaces the reference's thread-per-query knnGatherKernel with its fused
// covariance, the device eigen kernel and the projection kernels
// (src/index/SpatialIndexKernels.cu:716-1086, 1716-1769;
// src/stages/NeighborhoodKernels.cu:67-119, 422-485).
//
// Four kernels share the work.  k_knn_lane searches 64 queries per wave, one per
// lane, over one shared box of points staged in LDS; k_knn_pair the groups it
// finds too crowded, half a group at a time with two lanes per query.
// k_knn_group serves larger neighborhoods (and middling ones of small clouds)
// with one wave per query.  k_knn_rest searches the rows these leave, one per
// wave, with a box that grows around the row's own cell.  All find the fetch + 1
// smallest (d2, point id) pairs with the FP64 squared distances KD3Index
// computes (d0*d0 + d1*d1 + d2*d2, left to right, no FMA).
//
// Certification.  A query's list is exact when its fetch-th distance is below
// the distance from the query to the nearest face of the examined region
// (minus a rounding margin).  A query still uncertified when the growing
// box reaches the budget is flagged incomplete.  Rows whose fetch-th and
// (fetch+1)-th distances are equal have a boundary tie, which KD3Index breaks
// by tree visit order rather than by index; both kinds go to the exact KD3
// search.
//
// Covariance.  A row's FP64 covariance (two-pass mean) is formed by one lane
// from the kept list in (d2, id) order, the same sums in the same order in
// every kernel, and written in sorted order for the eigen/feature kernel.
#include "gf_eigen.hpp"
#include "gf_internal.hpp"
#include "gf_kernels.hpp"
#include "gf_stage.hpp"
#include "gf_wave.hpp"

namespace gf {

namespace {

constexpr uint32_t kLaneSmall = 8;     // columns of up to this many points are taken whole
constexpr int kRegBatches = 4;   // candidates of one row in registers, 64 a batch
constexpr uint32_t kRegCand = kRegBatches * 64;
constexpr int kGroupBatches = 4; // the same for the box a group of rows shares
constexpr uint32_t kGroupCand = kGroupBatches * 64;
constexpr int kRadBatches = 4;   // the same for a radius group's shared box
constexpr uint32_t kRadCand = kRadBatches * 64;
// Per-wave LDS scratch: 64 compacted entries (16 B) and 64 ranked entries.
constexpr int kScratchWords = 256 + 256;

// First positions in a[lo, hi) (sorted ascending) of keys >= k0 and of keys
// >= k1 (k0 <= k1): two binary searches advanced together, so that their
// loads are issued side by side (half the dependent load chain of running
// them one after the other).
__device__ __forceinline__ void lower_bound2_u32(const uint32_t* __restrict__ a, uint32_t lo,
                                                 uint32_t hi, uint32_t k0, uint32_t k1,
                                                 uint32_t& r0, uint32_t& r1)
{
    uint32_t lo0 = lo, hi0 = hi, lo1 = lo, hi1 = hi;
    while (lo0 < hi0 || lo1 < hi1) {
        const uint32_t m0 = lo0 + ((hi0 - lo0) >> 1), m1 = lo1 + ((hi1 - lo1) >> 1);
        const uint32_t v0 = lo0 < hi0 ? a[m0] : 0u;
        const uint32_t v1 = lo1 < hi1 ? a[m1] : 0u;
        if (lo0 < hi0) {
            if (v0 < k0)
                lo0 = m0 + 1;
            else
                hi0 = m0;
        }
        if (lo1 < hi1) {
            if (v1 < k1)
                lo1 = m1 + 1;
            else
                hi1 = m1;
        }
    }
    r0 = lo0;
    r1 = lo1;
}

// Block index -> logical block, so that each XCD (blocks are dealt to the 8
// XCDs round-robin) works on one contiguous run of sorted queries and its L2
// sees neighboring columns.
__device__ __forceinline__ uint32_t xcd_logical_block(uint32_t b, uint32_t nb)
{
    const uint32_t x = 8;
    uint32_t xcd = b % x, idx = b / x, per = nb / x, rem = nb % x;
    return xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

struct KnnArgs {
    CloudView cv;       // tiled: global arrays; colstart of all tiles
    FusedProgram prog;  // tiled: replaced per wave by the tile's
    KnnOutputs out;
    KnnTuning tune;
    int32_t mode;     // 0 features, 1 neighbor lists, 2 lists in KD3Index order
    int32_t q_per_wave;
    int32_t lds_stride;
    double margin;
    const TileInfo* tiles;   // tiled search only
    const uint64_t* starts;  // tiled: first row of each tile (ntiles + 1)
    const uint32_t* task0;   // tiled: per-tile first task (ntiles + 1)
    uint32_t ntasks;
    uint32_t ntiles;
    int32_t fetch_lo, fetch_hi;  // tiled: the result capacities this launch serves
    int32_t all_rows;        // k_knn_rest: every row instead of out.deferred
    int32_t group_q;         // k_knn_group: queries per wave (q_per_wave is a multiple)
    int32_t group_own;       // k_knn_group: a wave may search its left rows itself
};

// What a wavefront needs of its cloud or tile: the grid, the column starts,
// the certification margin and the neighborhood sizes.
struct WaveGrid {
    GridParams g;
    const uint32_t* colstart;
    double margin;
    int fetch, k, stride;
};

// The examined region: columns [x0, x1] x [y0, y1], z cells [z0, z1].
struct Box {
    int x0, x1, y0, y1, z0, z1;
};

// Distance from the query to the nearest face of the box that borders grid
// cells outside it (faces on the grid's edge bound nothing: +inf).
__device__ __forceinline__ double box_clearance(const GridParams& g, const Box& b,
                                                double qx, double qy, double qz)
{
    double R = INFINITY;
    if (b.x0 > 0) R = fmin(R, qx - (g.ox + static_cast<double>(b.x0) * g.c));
    if (b.x1 < static_cast<int>(g.gx) - 1)
        R = fmin(R, (g.ox + static_cast<double>(b.x1 + 1) * g.c) - qx);
    if (b.y0 > 0) R = fmin(R, qy - (g.oy + static_cast<double>(b.y0) * g.c));
    if (b.y1 < static_cast<int>(g.gy) - 1)
        R = fmin(R, (g.oy + static_cast<double>(b.y1 + 1) * g.c) - qy);
    if (b.z0 > 0) R = fmin(R, qz - (g.oz + static_cast<double>(b.z0) * g.cz));
    if (b.z1 < static_cast<int>(g.gz) - 1)
        R = fmin(R, (g.oz + static_cast<double>(b.z1 + 1) * g.cz) - qz);
    return R;
}

__device__ __forceinline__ bool certified(const WaveGrid& wg, const Box& b, const Ent& kth,
                                          double qx, double qy, double qz)
{
    const double R = box_clearance(wg.g, b, qx, qy, qz);
    if (R == INFINITY) return true;
    if (kth.d == kInfD) return false;
    const double Rm = R - wg.margin;
    return Rm > 0.0 && ent_d2(kth) < Rm * Rm;
}

// Column ranges of a box, one column per lane (box columns must be <= 64):
// lo / len of the column's sorted points restricted to z cells [z0, z1]
// (whole columns when the box spans every z cell or the column holds at most
// `small` points).
__device__ __forceinline__ void box_ranges(const KnnArgs& a, const WaveGrid& wg, const Box& b,
                                           int cb, int lane, uint32_t small, uint32_t& lo,
                                           uint32_t& len)
{
    const CloudView& cv = a.cv;
    const GridParams& g = wg.g;
    const int w = b.x1 - b.x0 + 1;
    const int ncb = w * (b.y1 - b.y0 + 1);
    const int ci = cb + lane;
    lo = 0;
    len = 0;
    if (ci >= ncb) return;
    const int cx = b.x0 + ci % w;
    const int cy = b.y0 + ci / w;
    if (cx < 0 || cy < 0 || cx >= static_cast<int>(g.gx) || cy >= static_cast<int>(g.gy))
        return;
    const bool zfull = b.z0 <= 0 && b.z1 >= static_cast<int>(g.gz) - 1;
    const uint32_t col = column_index(g, cx, cy);
    uint32_t b0 = wg.colstart[col], b1 = wg.colstart[col + 1];
    if (!zfull && b1 - b0 > small) {
        const uint32_t klo = (col << g.bz) + static_cast<uint32_t>(max(b.z0, 0));
        const uint32_t khi = (col << g.bz) + static_cast<uint32_t>(min(b.z1, static_cast<int>(g.gz) - 1) + 1);
        lower_bound2_u32(cv.keys, b0, b1, klo, khi, b0, b1);
    }
    lo = b0;
    len = b1 - b0;
}

// The same for a box of ncb <= kCols * 64 columns inside the grid, kCols
// columns per lane, their loads side by side: column starts first, then the
// z windows of columns of more than kLaneSmall points, all searched together.
template <int kCols>
__device__ __forceinline__ void box_columns(const KnnArgs& a, const WaveGrid& wg, const Box& b,
                                            int ncb, int lane, uint32_t (&lo)[kCols],
                                            uint32_t (&len)[kCols])
{
    const GridParams& g = wg.g;
    const int w = b.x1 - b.x0 + 1;
    const float inv_w = 1.0f / static_cast<float>(w);
    const bool zfull = b.z0 <= 0 && b.z1 >= static_cast<int>(g.gz) - 1;
    uint32_t col[kCols];
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
        lo[i] = len[i] = col[i] = 0;
        const int ci = i * 64 + lane;
        if (ci < ncb) {
            // ci / w: ci < 2^10, so the rounded quotient is exact
            const int cy = static_cast<int>((static_cast<float>(ci) + 0.5f) * inv_w);
            col[i] = column_index(g, static_cast<uint32_t>(b.x0 + ci - cy * w),
                                  static_cast<uint32_t>(b.y0 + cy));
            lo[i] = wg.colstart[col[i]];
            len[i] = wg.colstart[col[i] + 1];
        }
    }
#pragma unroll
    for (int i = 0; i < kCols; ++i) len[i] -= lo[i];
    if (zfull) return;
    bool tall = false;
#pragma unroll
    for (int i = 0; i < kCols; ++i) tall |= len[i] > kLaneSmall;
    if (!__ballot(tall)) return;
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
        if (len[i] > kLaneSmall) {
            const uint32_t klo = (col[i] << g.bz) + static_cast<uint32_t>(b.z0);
            const uint32_t khi = (col[i] << g.bz) + static_cast<uint32_t>(b.z1 + 1);
            uint32_t r0, r1;
            lower_bound2_u32(a.cv.keys, lo[i], lo[i] + len[i], klo, khi, r0, r1);
            lo[i] = r0;
            len[i] = r1 - r0;
        }
    }
}

// Sorted position of candidate t of the packed ranges: the lane whose range
// holds t is the last lane with excl <= t.
__device__ __forceinline__ uint32_t candidate_pos(uint32_t lo, uint32_t excl, uint32_t t)
{
    int src = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) {
        int p = src + step;
        uint32_t e = __shfl(excl, p & 63);
        if (p < 64 && e <= t) src = p;
    }
    const uint32_t slo = __shfl(lo, src);
    const uint32_t sex = __shfl(excl, src);
    return slo + (t - sex);
}

// Bit pattern of the FP64 squared distance, in KD3Index's operation order.
__device__ __forceinline__ uint64_t dist_bits(double qx, double qy, double qz, double px,
                                              double py, double pz)
{
    const double dx = qx - px;
    const double dy = qy - py;
    const double dz = qz - pz;
    double d2 = dx * dx;
    d2 = d2 + dy * dy;
    d2 = d2 + dz * dz;
    return static_cast<uint64_t>(__double_as_longlong(d2));
}

__device__ __forceinline__ double bits_d2(uint64_t d)
{
    return __longlong_as_double(static_cast<long long>(d));
}

__device__ __forceinline__ Ent make_ent(double qx, double qy, double qz, double px,
                                        double py, double pz, uint32_t id, uint32_t j)
{
    const double dx = qx - px;
    const double dy = qy - py;
    const double dz = qz - pz;
    double d2 = dx * dx;
    d2 = d2 + dy * dy;
    d2 = d2 + dz * dz;
    return Ent{static_cast<uint64_t>(__double_as_longlong(d2)), id, j};
}

// 1 when the compacted entry e = (d2 bits low, high, id, payload) precedes
// (d, id) in (d2, id) order.  Evaluated without branches, so that unrolled
// iterations issue their LDS loads together (short-circuit forms compile to
// one conditional load, and one wait, per entry).  Non-negative doubles order
// as their bit patterns.
__device__ __forceinline__ uint32_t rank_step(const uint4 e, uint64_t d, uint32_t id)
{
    const uint64_t od = static_cast<uint64_t>(e.x) | (static_cast<uint64_t>(e.y) << 32);
    return static_cast<uint32_t>(od < d) |
           (static_cast<uint32_t>(od == d) & static_cast<uint32_t>(e.z < id));
}

// Selection over at most kRegCand candidate entries held in registers.  First a threshold E with need <= #{d2 <= E} <= cap (need = fetch +
// 1, so the (fetch+1)-th entry that decides ties is kept), by bisection on
// d2, each trial counted exactly by ballots.  The survivors are compacted into
// LDS and ranked: each
// lane counts the survivors that precede its own entry in (d2, id) order,
// reading them as LDS broadcasts, and stores itself at that rank.  Every
// candidate with d2 equal to the boundary distance is below E, so the first
// fetch+1 ranked survivors are exactly the fetch+1 smallest (d2, id) pairs.
// When no such E exists (more than 64 points at one distance) the register
// batches are merged one by one with bitonic networks instead.
//
// The lane's candidate of register batch b is (cd[b], cid[b], cj[b]): squared
// distance bits (kInfD: none), point id and sorted position.
// (hint: a threshold to try first, as the previous query's need-th distance;
// INFINITY for none.)
template <int NB>
__device__ __forceinline__ void select_entries(const uint64_t (&cd)[NB],
                                               const uint32_t (&cid)[NB],
                                               const uint32_t (&cj)[NB], uint32_t tot,
                                               int fetch, int lane, uint32_t* scratch,
                                               double hint, Ent& best, uint64_t* cnt)
{
    const uint32_t need = min(static_cast<uint32_t>(fetch + 1), tot);
    // Survivor window: few enough to rank cheaply, at most one per lane.
    const uint32_t cap = min(need + 15u, 64u);
    bool ok = true;
    double E = INFINITY;
    cnt[2] += 1;
    if (tot > cap) {
        const uint32_t nbat = (tot + 63u) >> 6;  // register batches holding candidates
        auto count_le = [&](double t) {
            uint32_t k = 0;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (static_cast<uint32_t>(b) < nbat)
                    k += __popcll(__ballot(cd[b] != kInfD && bits_d2(cd[b]) <= t));
            return k;
        };
        ok = false;
        double lo_e = 0.0, hi_e = INFINITY;
        if (hint < INFINITY) {
            const uint32_t k = count_le(hint);
            if (k >= need && k <= cap) {
                E = hint;
                ok = true;
            } else if (k > cap) {
                hi_e = hint;
            } else {
                lo_e = hint;
            }
        }
        if (!ok && hi_e == INFINITY) {
            double mx = 0.0;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (static_cast<uint32_t>(b) < nbat && cd[b] != kInfD) mx = fmax(mx, bits_d2(cd[b]));
#pragma unroll
            for (int m = 32; m > 0; m >>= 1) mx = fmax(mx, __shfl_xor(mx, m));
            hi_e = mx;  // counts every candidate (> cap)
        }
        for (int it = 0; it < 80 && !ok; ++it) {
            const double mid = 0.5 * (lo_e + hi_e);
            const uint32_t k = count_le(mid);
            if (k < need) {
                if (!(mid > lo_e)) break;
                lo_e = mid;
            } else if (k > cap) {
                if (!(mid < hi_e)) break;
                hi_e = mid;
            } else {
                E = mid;
                ok = true;
            }
        }
    }
    if (ok) {
        uint32_t S = 0;
        const uint32_t nbat_s = (tot + 63u) >> 6;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if (static_cast<uint32_t>(b) >= nbat_s) break;
            const bool s = cd[b] != kInfD && bits_d2(cd[b]) <= E;
            const uint64_t m = __ballot(s);
            if (s) {
                // Survivors of lower lanes in this batch (mbcnt: popcount of
                // the ballot below this lane).
                const uint32_t below = __builtin_amdgcn_mbcnt_hi(
                    static_cast<uint32_t>(m >> 32),
                    __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
                uint32_t* e = scratch + 4 * (S + below);
                e[0] = static_cast<uint32_t>(cd[b]);
                e[1] = static_cast<uint32_t>(cd[b] >> 32);
                e[2] = cid[b];
                e[3] = cj[b];
            }
            S += __popcll(m);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        Ent v = ent_inf();
        uint32_t rank = 0;
        if (static_cast<uint32_t>(lane) < S) {
            const uint32_t* e = scratch + 4 * lane;
            v.d = static_cast<uint64_t>(e[0]) | (static_cast<uint64_t>(e[1]) << 32);
            v.id = e[2];
            v.j = e[3];
        }
#pragma unroll 4
        for (uint32_t i = 0; i < S; ++i)
            rank += rank_step(reinterpret_cast<const uint4*>(scratch)[i], v.d, v.id);
        uint32_t* sorted = scratch + 256;
        if (static_cast<uint32_t>(lane) < S) {
            uint32_t* e = sorted + 4 * rank;
            e[0] = static_cast<uint32_t>(v.d);
            e[1] = static_cast<uint32_t>(v.d >> 32);
            e[2] = v.id;
            e[3] = v.j;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        best = ent_inf();
        if (static_cast<uint32_t>(lane) < S) {
            const uint32_t* e = sorted + 4 * lane;
            best.d = static_cast<uint64_t>(e[0]) | (static_cast<uint64_t>(e[1]) << 32);
            best.id = e[2];
            best.j = e[3];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        return;
    }
    best = ent_inf();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (static_cast<uint32_t>(b * 64) >= tot) break;
        Ent c = cd[b] != kInfD ? Ent{cd[b], cid[b], cj[b]} : ent_inf();
        bitonic_sort64(c, lane);
        merge_sorted(best, c, lane);
        cnt[2] += 1;
    }
}

// Candidates whose d2 bits are <= t (below t when kStrict); kInfD entries
// never count.  Non-negative doubles order as their bit patterns.
template <bool kStrict>
__device__ __forceinline__ uint32_t count_bits(const uint64_t (&cd)[kGroupBatches], uint32_t nbat,
                                               uint64_t t)
{
    uint32_t c = 0;
#pragma unroll
    for (int b = 0; b < kGroupBatches; ++b)
        if (static_cast<uint32_t>(b) < nbat)
            c += __popcll(__ballot(kStrict ? cd[b] < t : cd[b] <= t));
    return c;
}

__device__ __forceinline__ uint64_t d2_bits(double d)
{
    return static_cast<uint64_t>(__double_as_longlong(d));
}

// Exact-count selection, for neighborhoods kept as a set (features, stride
// 1): a threshold E with exactly `fetch` candidates at d2 <= E.  Such an E
// exists exactly when the fetch-th and (fetch+1)-th smallest distances
// differ (no boundary tie), and the kept set is then {d2 <= E} whatever the
// order among equal distances inside it.  Counts are exact (ballots).  First
// round: kRound thresholds around the hint (the previous query's E) counted
// together; one with count fetch is E, else the two around fetch bracket it,
// and when few candidates lie inside the bracket each ranks itself among
// them and the one at the wanted rank, checked by its count, is E.  Failing
// that: linear interpolation of the count in d2 inside the bracket, then
// candidates strictly inside it as pivots.  A bracket with no candidate
// strictly inside means the fetch-th and (fetch+1)-th distances are equal:
// false, and the caller takes the sorting selection (as when the trials run
// out).
//
// Thresholds of the first round, as factors of the hint (for points on a
// surface the count grows about linearly with d2).
constexpr int kRound = 7;

__device__ __forceinline__ float round_factor(int i)
{
    constexpr float f[kRound] = {0.6f, 0.75f, 0.87f, 1.0f, 1.15f, 1.33f, 1.6f};
    return f[i];
}

__device__ __forceinline__ bool select_count(const uint64_t (&cd)[kGroupBatches], uint32_t nbat,
                                             uint32_t fetch, double hint, uint64_t& E)
{
    const double h = uniform_f64(hint);
    // First round: counts at kRound thresholds around the hint, independent
    // of each other (one latency for all of them).
    uint64_t tb[kRound];
    uint32_t c[kRound];
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
        tb[i] = d2_bits(h * static_cast<double>(round_factor(i)));
        c[i] = 0;
    }
#pragma unroll
    for (int b = 0; b < kGroupBatches; ++b) {
        if (static_cast<uint32_t>(b) >= nbat) break;
#pragma unroll
        for (int i = 0; i < kRound; ++i) c[i] += __popcll(__ballot(cd[b] <= tb[i]));
    }
    // The bracket: the last threshold below fetch, the first above.
    int ilo = -1, ihi = kRound;
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
        if (c[i] == fetch) {
            E = tb[i];
            return true;
        }
        if (c[i] < fetch) ilo = i;
        if (c[i] > fetch && ihi == kRound) ihi = i;
    }
    double lo = 0.0, hi = INFINITY;
    uint32_t clo = 0, chi = 0;
    uint64_t lob = 0, hib = kInfD;
#pragma unroll
    for (int i = 0; i < kRound; ++i) {
        if (i == ilo) {
            lob = tb[i];
            clo = c[i];
        }
        if (i == ihi) {
            hib = tb[i];
            chi = c[i];
        }
    }
    if (ilo >= 0) lo = bits_d2(lob);
    if (ihi < kRound) hi = bits_d2(hib);
    if (ihi < kRound && chi - clo <= 16u) {
        // Few candidates inside the bracket: each ranks itself among them
        // (strictly smaller ones), and the one at rank fetch - clo - 1 is the
        // fetch-th distance when it is alone there; checked by its count.
        uint64_t mb[kGroupBatches];
        uint32_t rk[kGroupBatches];
#pragma unroll
        for (int b = 0; b < kGroupBatches; ++b) {
            rk[b] = 0;
            mb[b] = static_cast<uint32_t>(b) < nbat
                        ? __ballot((ilo < 0 || cd[b] > lob) && cd[b] <= hib)
                        : 0ull;
        }
#pragma unroll
        for (int b = 0; b < kGroupBatches; ++b) {
            uint64_t m = mb[b];
            while (m) {
                const int l = __builtin_ctzll(m);
                m &= m - 1;
                const uint64_t v = lane_u64(cd[b], l);
#pragma unroll
                for (int b2 = 0; b2 < kGroupBatches; ++b2)
                    if (static_cast<uint32_t>(b2) < nbat) rk[b2] += v < cd[b2] ? 1u : 0u;
            }
        }
        const uint32_t want = fetch - clo - 1;
        uint64_t pick = kInfD;
        uint32_t npick = 0;
#pragma unroll
        for (int b = 0; b < kGroupBatches; ++b) {
            if (static_cast<uint32_t>(b) >= nbat) break;
            const uint64_t m = mb[b] & __ballot(rk[b] == want);
            npick += static_cast<uint32_t>(__popcll(m));
            if (m && pick == kInfD) pick = lane_u64(cd[b], __builtin_ctzll(m));
        }
        if (npick == 1) {
            if (count_bits<false>(cd, nbat, pick) == fetch) {
                E = pick;
                return true;
            }
        }
    }
    // Otherwise: linear interpolation of the count in d2 inside the bracket,
    // then candidates strictly inside the bracket as pivots.  When the
    // bracket holds no candidate strictly inside, the fetch-th and
    // (fetch+1)-th distances are equal: false.
    double t;
    if (hi == INFINITY) {
        t = (ilo >= 0 ? lo : h) * static_cast<double>((static_cast<float>(fetch) + 0.5f) /
                                                    static_cast<float>(clo > 0 ? clo : 1));
    } else {
        const float f = (static_cast<float>(fetch - clo) + 0.5f) / static_cast<float>(chi - clo);
        t = lo + (hi - lo) * static_cast<double>(f);
    }
#pragma unroll 1
    for (int trial = 0; trial < 16; ++trial) {
        if (trial >= 3 || !(t > lo && t < hi)) {
            // Pivot: the first candidate strictly inside (lo, hi).
            const uint64_t lb = d2_bits(lo), hb = d2_bits(hi);
            uint64_t piv = kInfD;
#pragma unroll
            for (int b = 0; b < kGroupBatches; ++b) {
                if (static_cast<uint32_t>(b) >= nbat || piv != kInfD) continue;
                const uint64_t m = __ballot(cd[b] > lb && cd[b] < hb);
                if (m) piv = lane_u64(cd[b], __builtin_ctzll(m));
            }
            if (piv == kInfD) return false;
            t = bits_d2(piv);
        }
        const uint64_t tbt = d2_bits(t);
        const uint32_t ct = count_bits<false>(cd, nbat, tbt);
        if (ct == fetch) {
            E = tbt;
            return true;
        }
        if (ct < fetch) {
            lo = t;
            clo = ct;
        } else {
            hi = t;
            chi = ct;
        }
        if (hi == INFINITY) {
            // Count ~ d2 through the origin.
            t = lo * static_cast<double>((static_cast<float>(fetch) + 0.5f) /
                                         static_cast<float>(clo > 0 ? clo : 1));
        } else {
            const float f = (static_cast<float>(fetch - clo) + 0.5f) /
                            static_cast<float>(chi - clo);
            t = lo + (hi - lo) * static_cast<double>(f);
        }
    }
    return false;
}

// Lane l's value of v, for every lane (l wave-uniform).
__device__ __forceinline__ double lane_value(double v, int l)
{
    const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(b), l);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(b >> 32), l);
    return __longlong_as_double(
        static_cast<long long>(static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32)));
}

__device__ __forceinline__ uint32_t lanes_below64(uint64_t m)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u));
}

// The n (<= 64) entries waiting in scratch, sorted and merged into best.
__device__ __forceinline__ void stream_flush(const uint32_t* scratch, uint32_t n, int lane,
                                             Ent& best)
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    Ent c = ent_inf();
    if (static_cast<uint32_t>(lane) < n) {
        const uint32_t* e = scratch + 4 * lane;
        c.d = static_cast<uint64_t>(e[0]) | (static_cast<uint64_t>(e[1]) << 32);
        c.id = e[2];
        c.j = e[3];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    bitonic_sort64(c, lane);
    merge_sorted(best, c, lane);
}

// One query alone, with a growing box starting at half-width r (columns and
// z cells around the query's cell): candidates stream through the registers
// (<= 256, one box of <= 64 columns) or through sort-and-merge otherwise.
__device__ __forceinline__ void search_single(const KnnArgs& a, const WaveGrid& wg, double qx,
                              double qy, double qz, int qcx, int qcy, int qcz, int r, int lane,
                              uint32_t* scratch, Ent& best, bool& incomplete,
                              uint64_t* cnt)
{
    const CloudView& cv = a.cv;
    const int fetch = wg.fetch;
    incomplete = false;
    uint32_t nbuf = 0;  // streamed candidates waiting in LDS
    for (;;) {
        cnt[0] += 1;
        const Box b{qcx - r, qcx + r, qcy - r, qcy + r, qcz - r, qcz + r};
        const int ncb = (2 * r + 1) * (2 * r + 1);
        best = ent_inf();
        for (int cb = 0; cb < ncb; cb += 64) {
            uint32_t lo, len;
            box_ranges(a, wg, b, cb, lane, static_cast<uint32_t>(a.tune.small_col), lo, len);
            const uint32_t incl = wave_incl_scan_u32(len, lane);
            const uint32_t tot = lane_u32(incl, 63);
            const uint32_t excl = incl - len;
            cnt[1] += tot;
            if (ncb <= 64 && tot <= kRegCand) {
                uint64_t cd[kRegBatches];
                uint32_t cid[kRegBatches], cj[kRegBatches];
#pragma unroll
                for (int bb = 0; bb < kRegBatches; ++bb) {
                    cd[bb] = kInfD;
                    cid[bb] = cj[bb] = kInfU;
                    if (static_cast<uint32_t>(bb * 64) < tot) {
                        const uint32_t t = bb * 64 + lane;
                        const uint32_t j = candidate_pos(lo, excl, t);
                        if (t < tot) {
                            cd[bb] = dist_bits(qx, qy, qz, cv.sx[j], cv.sy[j], cv.sz[j]);
                            cid[bb] = cv.perm[j];
                            cj[bb] = j;
                        }
                    }
                }
                select_entries(cd, cid, cj, tot, fetch, lane, scratch, INFINITY, best, cnt);
                break;
            }
            // Streamed: candidates below the current (fetch+1)-th entry are
            // collected in LDS and sorted into the list 64 at a time.  That
            // entry only decreases, so a candidate not below it when it
            // is seen cannot be among the final fetch+1.
            for (uint32_t t0 = 0; t0 < tot; t0 += 64) {
                const uint32_t t = t0 + lane;
                const uint32_t j = candidate_pos(lo, excl, t);
                Ent c = ent_inf();
                if (t < tot)
                    c = make_ent(qx, qy, qz, cv.sx[j], cv.sy[j], cv.sz[j], cv.perm[j], j);
                const Ent worst = ent_lane(best, fetch);
                const bool surv = t < tot && ent_less(c, worst);
                const uint64_t m = __ballot(surv);
                if (!m) continue;
                const uint32_t ns = static_cast<uint32_t>(__popcll(m));
                if (nbuf + ns > 64u) {
                    stream_flush(scratch, nbuf, lane, best);
                    cnt[2] += 1;
                    nbuf = 0;
                }
                if (surv) {
                    uint32_t* e = scratch + 4 * (nbuf + lanes_below64(m));
                    e[0] = static_cast<uint32_t>(c.d);
                    e[1] = static_cast<uint32_t>(c.d >> 32);
                    e[2] = c.id;
                    e[3] = c.j;
                }
                nbuf += ns;
            }
        }
        if (nbuf) {
            stream_flush(scratch, nbuf, lane, best);
            cnt[2] += 1;
            nbuf = 0;
        }
        const Ent kth = ent_lane(best, fetch - 1);
        if (certified(wg, b, kth, qx, qy, qz)) return;
        if (r >= a.tune.ring_max) {
            incomplete = true;
            return;
        }
        int rn = r + 1;
        if (kth.d != kInfD) {
            const double rr = ceil((sqrt(ent_d2(kth)) + wg.margin) / wg.g.c);
            if (rr > rn) rn = rr > 1e6 ? 1000000 : static_cast<int>(rr);
        } else {
            rn = max(rn, 2 * r);
        }
        r = min(rn, a.tune.ring_max);
    }
}

// Tie test and hand-off of one query's result: in neighbor-list mode the kept
// ids go straight to global memory; in feature mode the kept sorted positions
// are parked in LDS for the covariance pass.
__device__ __forceinline__ void finish_query(const KnnArgs& a, const WaveGrid& wg, const Ent& best,
                                             bool incomplete, uint64_t s, int qslot,
                                             int lane, uint32_t* nbr, uint8_t& my_flags)
{
    const int fetch = wg.fetch;
    const int k = wg.k;
    const int stride = wg.stride;
    // Boundary tie: the fetch-th and (fetch+1)-th distances are equal.  With
    // stride > 1 every adjacent equal pair inside the fetched list can change
    // which ids are kept, and ordered lists (mode 2) need KD3Index's order
    // among equal distances, so there any such pair flags the row.
    const Ent nxt = ent_shfl(best, lane + 1 < 64 ? lane + 1 : 63);
    const bool eq = (lane < fetch) && (lane + 1 < 64) && best.d == nxt.d && best.d != kInfD;
    const bool tie = (stride > 1 || a.mode == 2)
                         ? (__ballot(eq) != 0)
                         : (lane_u32(eq ? 1u : 0u, fetch - 1) != 0);
    const uint8_t flags = (tie ? ST_TIE : 0) | (incomplete ? ST_INCOMPLETE : 0);
    // Kept list in canonical (d2, id) order: entries 0, stride, 2*stride...
    const Ent kept = ent_shfl(best, (lane * stride) & 63);
    if (a.mode != 0) {
        const uint32_t qid = a.cv.perm[s];
        // Mode 2 keeps sorted positions (the consumer reads the sorted
        // coordinates, which neighbors share cache lines in).
        if (lane < k)
            a.out.ids[static_cast<uint64_t>(qid) * k + lane] = a.mode == 2 ? kept.j : kept.id;
        if (lane == 0) a.out.status[0][qid] = flags;
        if (lane == 0 && flags) {
            uint32_t slot = atomicAdd(a.out.nflagged, 1u);
            a.out.flagged[slot] = static_cast<uint32_t>(s);
            atomicAdd(a.out.nflagged + ((flags & ST_INCOMPLETE) ? 2 : 1), 1u);
        }
    } else {
        // An uncertified row can hold fewer than fetch entries; keep its list
        // in bounds (the exact search replaces the row).
        if (lane < k) nbr[qslot * a.lds_stride + lane] = kept.j == kInfU ? 0u : kept.j;
        if (lane == qslot) my_flags = flags;
    }
}

// The tile holding sorted row s.
__device__ __forceinline__ uint32_t tile_of(const uint64_t* __restrict__ starts, uint32_t T,
                                            uint64_t s)
{
    uint32_t lo = 0, hi = T;  // largest t with starts[t] <= s
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (starts[mid] <= s)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

__device__ __forceinline__ void tile_grid(const KnnArgs& a, const TileInfo& ti, WaveGrid& wg)
{
    wg.g = ti.g;
    wg.colstart = a.cv.colstart + ti.colbase;
    wg.margin = ti.margin;
    wg.fetch = ti.prog.fetch;
    wg.k = ti.prog.k;
    wg.stride = ti.prog.stride;
}

__device__ __forceinline__ void cloud_grid(const KnnArgs& a, WaveGrid& wg)
{
    wg.g = a.cv.g;
    wg.colstart = a.cv.colstart;
    wg.margin = a.margin;
    wg.fetch = a.prog.fetch;
    wg.k = a.prog.k;
    wg.stride = a.prog.stride;
}

// The wave's queries [q0, q0 + nq) and its cloud's or tile's grid and
// program; false for a task past the last one.
template <bool kTiled>
__device__ __forceinline__ bool wave_queries(const KnnArgs& a, uint64_t task, int Q, WaveGrid& wg,
                                             uint64_t& q0, int& nq)
{
    if (kTiled) {
        if (task >= a.ntasks) return false;
        // The task's tile: the last t with task0[t] <= task (tiles with no
        // task share the next tile's prefix).
        uint32_t tlo = 0, thi = a.ntiles;
        while (thi - tlo > 1) {
            const uint32_t mid = (tlo + thi) >> 1;
            if (a.task0[mid] <= task)
                tlo = mid;
            else
                thi = mid;
        }
        const TileInfo& ti = a.tiles[tlo];
        const uint64_t first = (task - a.task0[tlo]) * static_cast<uint64_t>(Q);
        tile_grid(a, ti, wg);
        q0 = ti.start + first;
        nq = static_cast<int>(ti.n - first < static_cast<uint64_t>(Q) ? ti.n - first : Q);
        return true;
    }
    cloud_grid(a, wg);
    q0 = task * static_cast<uint64_t>(Q);
    if (q0 >= a.cv.n) return false;
    nq = static_cast<int>(a.cv.n - q0 < static_cast<uint64_t>(Q) ? a.cv.n - q0 : Q);
    return true;
}

// ------------------------------------------------- query-per-lane search --
//
// A wave takes Q (<= 64) consecutive sorted queries, one per lane.  The
// queries' bounding box grown by a search radius r is staged once in LDS: the
// FP64 coordinates and sorted positions of the points inside it,
// counting-sorted into small cells (x fastest), so that the cells a query can
// see in one row are one contiguous run.  Every lane then walks its own runs
// -- the rows (and, in tall boxes, layers) within its own radius rl <= r,
// chosen from the number of points around it -- computes KD3Index's FP64
// squared distances and appends (distance, slot) to its own list when below
// its bound E (at first rl * rl).  A list that fills up is sorted in registers
// (a compile-time merge-exchange network over 32-bit keys: the distance as
// FP32 without its low bits, the slot in their place) and cut back to the
// fetch + 1 + kLaneSlack smallest, and the bound drops to the largest of them.
//
// The 32-bit keys only order coarsely; at the end the kept entries' FP64
// distances are put into (d2, id) order exactly.  A row is final when its
// fetch-th distance is below its radius squared and its (fetch + 1)-th below
// every entry cut away.  The radius is at most the ring_max cells that bound
// the growing search, so a row found here is one that search would certify.
// A group whose box holds too many points is halved along its longest axis.
// A few lanes not final go to k_knn_rest; more of them are tried again with
// a larger radius first.
//
// Bound by vector instructions (staging, walks and the sorting network) at the
// five to seven waves per CU that their LDS allows (22.0, 26.0 and 30.0 KB by
// instance), so that some SIMDs hold two: hence at most 256 registers.  Against
// the wave-per-query search for every row, search time: 4M points k 16 8.4 -> 5.2
// ms, 777k k 8 stride 3 3.6 -> 2.2, 250k k 10 1.67 -> 0.63; 10M points of terrain
// and flat roofs, k 32, 34 -> 27.
constexpr int kLaneSlack = 2;   // entries beyond fetch + 1 put in exact order
// First radius over the one the density's estimate gives, and the points a
// lane's radius should hold over fetch + 1 (measured best of 1.2 to 1.7 and 1.5
// to 2.1: smaller ones fail lanes, larger ones fill boxes and lists).
constexpr float kRadiusFactor = 1.35f;
constexpr float kListFactor = 1.8f;
constexpr int kLaneFew = 6;     // lanes not worth another round of their own
constexpr uint32_t kStageMax = 512;    // points staged per round
constexpr int kStageSlots = 16;        // points of the box's columns per lane and round
constexpr uint32_t kStageRaw = kStageSlots * 64;
constexpr uint32_t kStageCells = 512;
constexpr int kStageCols = 5;          // columns of a box per lane
constexpr int kListRow = 65;    // LDS words between list positions of the ordered lists
static_assert(kStageMax <= kSlotMask + 1);  // a slot fits a key's low bits

template <int P, int Q, int R, int D, int N>
__device__ __forceinline__ void sort_step(uint32_t (&k)[N])
{
#pragma unroll
    for (int i = 0; i < N - D; ++i)
        if ((i & P) == R) {
            const uint32_t a = min(k[i], k[i + D]), b = max(k[i], k[i + D]);
            k[i] = a;
            k[i + D] = b;
        }
    if constexpr (Q != P) sort_step<P, Q / 2, P, Q - P, N>(k);
}

template <int P, int T, int N> __device__ __forceinline__ void sort_phase(uint32_t (&k)[N])
{
    if constexpr (P > 0) {
        sort_step<P, T, 0, P, N>(k);
        sort_phase<P / 2, T, N>(k);
    }
}

constexpr int half_pow2(int n)  // largest power of two below n
{
    int t = 1;
    while (2 * t < n) t *= 2;
    return t;
}

// Ascending sort of N registers (Knuth's merge exchange, algorithm 5.2.2M).
template <int N> __device__ __forceinline__ void sort_net(uint32_t (&k)[N])
{
    constexpr int T = half_pow2(N);
    sort_phase<T, T, N>(k);
}

// Reductions and scans over the whole wave by data-parallel moves within the
// register file (rows of 16 lanes, then the rows' last lanes); every lane
// must be active.
template <int kCtrl, int kRows> __device__ __forceinline__ uint32_t dpp_u32(uint32_t old, uint32_t v)
{
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
        static_cast<int>(old), static_cast<int>(v), kCtrl, kRows, 0xF, false));
}

__device__ __forceinline__ float wave_min_f32(float v)
{
    auto step = [&](uint32_t o) { v = fminf(v, __uint_as_float(o)); };
    step(dpp_u32<0x111, 0xF>(__float_as_uint(v), __float_as_uint(v)));
    step(dpp_u32<0x112, 0xF>(__float_as_uint(v), __float_as_uint(v)));
    step(dpp_u32<0x114, 0xF>(__float_as_uint(v), __float_as_uint(v)));
    step(dpp_u32<0x118, 0xF>(__float_as_uint(v), __float_as_uint(v)));
    step(dpp_u32<0x142, 0xA>(__float_as_uint(v), __float_as_uint(v)));
    step(dpp_u32<0x143, 0xC>(__float_as_uint(v), __float_as_uint(v)));
    return __uint_as_float(lane_u32(__float_as_uint(v), 63));
}

// Extent of v over the active lanes of the first and second half of the
// wave's queries: halves of the wave, or (two lanes per query) of its first
// half.
template <int LPQ> __device__ __forceinline__ float2 half_extents(bool act, float v)
{
    float lo = act ? v : INFINITY, hi = act ? -v : INFINITY;
    auto step = [&](float& m, uint32_t o) { m = fminf(m, __uint_as_float(o)); };
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float& m = i ? hi : lo;
        step(m, dpp_u32<0x111, 0xF>(__float_as_uint(m), __float_as_uint(m)));
        step(m, dpp_u32<0x112, 0xF>(__float_as_uint(m), __float_as_uint(m)));
        step(m, dpp_u32<0x114, 0xF>(__float_as_uint(m), __float_as_uint(m)));
        step(m, dpp_u32<0x118, 0xF>(__float_as_uint(m), __float_as_uint(m)));
        if (LPQ == 1) step(m, dpp_u32<0x142, 0xA>(__float_as_uint(m), __float_as_uint(m)));
    }
    const float e = -hi - lo;
    return make_float2(__uint_as_float(lane_u32(__float_as_uint(e), LPQ == 1 ? 31 : 15)),
                       __uint_as_float(lane_u32(__float_as_uint(e), LPQ == 1 ? 63 : 31)));
}

__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v)
{
    v += dpp_u32<0x111, 0xF>(0u, v);
    v += dpp_u32<0x112, 0xF>(0u, v);
    v += dpp_u32<0x114, 0xF>(0u, v);
    v += dpp_u32<0x118, 0xF>(0u, v);
    v += dpp_u32<0x142, 0xA>(0u, v);
    v += dpp_u32<0x143, 0xC>(0u, v);
    return v;
}

// The lane's list (LDS, one column per lane), sorted; its entries after cnt
// read as the largest key.
template <int CAP>
__device__ __forceinline__ void load_sorted(const uint32_t* my, uint32_t cnt, uint32_t (&k)[CAP])
{
#pragma unroll
    for (int i = 0; i < CAP; ++i) {
        const uint32_t v = my[i * 64];
        k[i] = static_cast<uint32_t>(i) < cnt ? v : kInfU;
    }
    sort_net<CAP>(k);
}

template <int CAP> struct StageShared {
    static constexpr bool kPositions = true;
    double x[kStageMax], y[kStageMax], z[kStageMax];
    uint32_t j[kStageMax];
    uint32_t cell[kStageCells + 2];   // counts, then first slots; last: points left out
    union {
        uint32_t list[CAP * 64];      // one list column per lane
        uint32_t pos[kStageRaw];      // while staging: sorted positions of the box's columns
    };
};

// stage_size for a box that every lane holds.
__device__ __forceinline__ bool size_box(StageBox& B, float r)
{
    const bool ok = stage_size(B, r, kStageCells);
    B.nx = uniform_i32(B.nx);
    B.ny = uniform_i32(B.ny);
    B.nz = uniform_i32(B.nz);
    return ok;
}

__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Stages the points of N <= kStageRaw column entries (lo, len: the lane's
// columns; at: entries of the lanes before it) that lie inside B's faces,
// counting-sorted by cell.  False if there are more than kStageMax.
template <class Shared>
__device__ __forceinline__ bool stage_points(const CloudView& cv, Shared& S,
                                             const uint32_t (&lo)[kStageCols],
                                             const uint32_t (&len)[kStageCols], uint32_t at,
                                             uint32_t N, const StageBox& B, int lane)
{
    // The columns' points, one per lane and slot.
#pragma unroll
    for (int i = 0; i < kStageCols; ++i)
        for (uint32_t c = 0; c < len[i]; ++c) S.pos[at++] = lo[i] + c;
#pragma unroll
    for (uint32_t c = 0; c < kStageCells; c += 64) S.cell[c + lane] = 0;
    wave_lds_order();
    // Four points per lane at a time; the coordinates are read
    // again (from cache) when the slots are known, so that
    // they do not hold registers in between.
    uint32_t pc[kStageSlots];  // cell << 16 | rank in it, or ~0
#pragma unroll
    for (int i0 = 0; i0 < kStageSlots; i0 += 4) {
        if (i0 * 64u >= N) {  // wave-uniform
#pragma unroll
            for (int i = 0; i < 4; ++i) pc[i0 + i] = ~0u;
            continue;
        }
        double px[4], py[4], pz[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = (i0 + i) * 64u + lane;
            const uint32_t j = S.pos[t < N ? t : 0u];
            px[i] = cv.sx[j];
            py[i] = cv.sy[j];
            pz[i] = cv.sz[j];
        }
        uint32_t cell[4], rank[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = (i0 + i) * 64u + lane;
            const int ix = min(static_cast<int>(static_cast<float>(px[i] - B.X0) * B.hx), B.nx - 1);
            const int iy = min(static_cast<int>(static_cast<float>(py[i] - B.Y0) * B.hy), B.ny - 1);
            const int iz = min(static_cast<int>(static_cast<float>(pz[i] - B.Z0) * B.hz), B.nz - 1);
            const bool in = static_cast<int>(t < N) & static_cast<int>(px[i] >= B.X0) &
                            static_cast<int>(px[i] <= B.X1) & static_cast<int>(py[i] >= B.Y0) &
                            static_cast<int>(py[i] <= B.Y1) & static_cast<int>(pz[i] >= B.Z0) &
                            static_cast<int>(pz[i] <= B.Z1);
            // (points outside count in a cell of their own)
            cell[i] = in ? static_cast<uint32_t>((iz * B.ny + iy) * B.nx + ix) : kStageCells + 1u;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) rank[i] = atomicAdd(&S.cell[cell[i]], 1u);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            pc[i0 + i] = cell[i] <= kStageCells ? (cell[i] << 16) | rank[i] : ~0u;
    }
    wave_lds_order();
    // First slots of the cells (eight cells per lane).
    constexpr int kPer = kStageCells / 64;
    uint32_t v[kPer], sum = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        v[i] = S.cell[lane * kPer + i];
        sum += v[i];
    }
    uint32_t ex = wave_scan_u32(sum);
    const uint32_t M = lane_u32(ex, 63);
    ex -= sum;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        S.cell[lane * kPer + i] = ex;
        ex += v[i];
    }
    if (lane == 0) S.cell[kStageCells] = M;
    wave_lds_order();
    if (M > kStageMax) return false;
#pragma unroll
    for (int i0 = 0; i0 < kStageSlots; i0 += 4) {
        if (i0 * 64u >= N) break;
        double px[4], py[4], pz[4];
        uint32_t j[4], at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = (i0 + i) * 64u + lane;
            j[i] = S.pos[t < N ? t : 0u];
            px[i] = cv.sx[j[i]];
            py[i] = cv.sy[j[i]];
            pz[i] = cv.sz[j[i]];
            const uint32_t c = pc[i0 + i];
            at[i] = c != ~0u ? S.cell[c >> 16] + (c & 0xFFFFu) : ~0u;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (at[i] != ~0u) {
                S.x[at[i]] = px[i];
                S.y[at[i]] = py[i];
                S.z[at[i]] = pz[i];
                if constexpr (Shared::kPositions) S.j[at[i]] = j[i];
            }
        }
    }
    wave_lds_order();
    return true;
}

// FP64 covariance of the k neighbors pos(0..k-1) (indexes into x, y, z;
// two-pass mean) into sorted row s's record, with its search flags.  Coordinates are taken
// relative to the query point (exact differences at any offset), so the mean
// carries no rounding of the cloud's absolute position: at UTM scale that
// rounding (~1e-9 m) would add a rank-one term to the covariance of flat and
// collinear neighborhoods.
template <class Pos>
__device__ __forceinline__ void write_cov_record(const KnnArgs& a, uint64_t s, int k, double ox,
                                                 double oy, double oz, uint8_t flags,
                                                 const double* x, const double* y,
                                                 const double* z, Pos pos)
{
    double mx = 0.0, my = 0.0, mz = 0.0;
#pragma unroll 4
    for (int l = 0; l < k; ++l) {
        const uint32_t j = pos(l);
        mx += x[j] - ox;
        my += y[j] - oy;
        mz += z[j] - oz;
    }
    mx /= static_cast<double>(k);
    my /= static_cast<double>(k);
    mz /= static_cast<double>(k);
    double c[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll 4
    for (int l = 0; l < k; ++l) {
        const uint32_t j = pos(l);
        const double dx = (x[j] - ox) - mx, dy = (y[j] - oy) - my,
                     dz = (z[j] - oz) - mz;
        c[0] += dx * dx;
        c[1] += dx * dy;
        c[2] += dx * dz;
        c[3] += dy * dy;
        c[4] += dy * dz;
        c[5] += dz * dz;
    }
    const double den = static_cast<double>(k - 1);
    double* rec = a.out.cov + kCovRecord * s;
    for (int i = 0; i < 6; ++i) rec[i] = c[i] / den;
    reinterpret_cast<uint64_t*>(rec)[6] = flags;
}

// The final rows of a wave: lists of slots (LDS, 65 words between positions,
// so that lanes read a position and rows read a list without bank conflicts)
// to covariance records or to the output lists.
__device__ __forceinline__ void store_rows(const KnnArgs& a, const WaveGrid& wg, uint64_t s,
                                           int lane, bool done, bool tie, double qx, double qy,
                                           double qz, const double* x, const double* y,
                                           const double* z, const uint32_t* sj,
                                           const uint32_t* list)
{
    const uint64_t dm = __ballot(done);
    if (!dm) return;
    const uint8_t flags = tie ? ST_TIE : 0;
    const int stride = wg.stride;
    if (a.mode == 0) {
        if (done)
            write_cov_record(a, s, wg.k, qx, qy, qz, flags, x, y, z,
                             [&](int l) { return list[l * stride * kListRow + lane]; });
    } else {
        const uint32_t qid = done ? a.cv.perm[s] : 0u;
        if (done) a.out.status[0][qid] = flags;
        // One row after another, its k entries side by side.
        for (uint64_t m = dm; m; m &= m - 1) {
            const int r = __builtin_ctzll(m);
            const uint64_t row = lane_u32(qid, r);
            if (lane < wg.k) {
                const uint32_t j = sj[list[lane * stride * kListRow + r]];
                a.out.ids[row * static_cast<uint64_t>(wg.k) + lane] =
                    a.mode == 2 ? j : a.cv.perm[j];
            }
        }
    }
    const uint64_t tm = __ballot(done && tie);
    if (tm) {
        uint32_t at = 0;
        if (lane == 0) {
            const uint32_t c = static_cast<uint32_t>(__popcll(tm));
            at = atomicAdd(a.out.nflagged, c);
            atomicAdd(a.out.nflagged + 1, c);
        }
        at = lane_u32(at, 0) + lanes_below64(tm);
        if (done && tie) a.out.flagged[at] = static_cast<uint32_t>(s);
    }
}

// The search of one group of queries [q0, q0 + nq); LPQ lanes per query (the
// second lane of a pair takes every other candidate, and the pair's two
// lists are merged before the exact order).  With kBail a group whose first
// box holds too many points is left whole: returns true, nothing written.
template <int CAP, int TM, int LPQ, bool kBail>
__device__ __forceinline__ bool search_group(const KnnArgs& a, const WaveGrid& wg, uint64_t q0,
                                             int nq, StageShared<CAP>& S)
{
    const int lane = __lane_id();
    const int ql = lane & (64 / LPQ - 1);  // the lane's query
    const int part = LPQ == 1 ? 0 : lane >> 5;
    const CloudView& cv = a.cv;
    const GridParams& g = wg.g;
    const uint32_t fetch = static_cast<uint32_t>(wg.fetch);
    const uint32_t keep = fetch + 1 + kLaneSlack;  // <= TM
    const bool valid = ql < nq;
    const uint64_t s = valid ? cv.qord[q0 + ql] : q0;
    const double qx = valid ? cv.sx[s] : 0.0;
    const double qy = valid ? cv.sy[s] : 0.0;
    const double qz = valid ? cv.sz[s] : 0.0;
    const uint32_t key0 = cv.keys[uniform_u32(cv.qord[q0])];
    uint32_t* my = S.list + lane;
    // The growing search's box reaches ring_max whole cells from a query's
    // own cell on every side.
    const double reach = static_cast<double>(a.tune.ring_max) * fmin(g.c, g.cz);
    const float r_cap = static_cast<float>((reach - 4.0 * wg.margin) * (1.0 - 1e-6));
    bool pending = valid && stage_takes(reach, wg.margin) && stage_takes_point(qx, qy, qz);
    bool defer = valid && !pending;
    uint32_t tries = 0;
    float r_need = 0.0f;  // the smallest radius worth trying for this lane
    // The first radius, from two densities around the wave: of a surface (the
    // first query's 8 x 8 columns), and of a volume (the denser half of the
    // wave's queries in its bounding box).
    float r_first = r_cap;
    {
        const uint32_t t = (key0 >> g.bz) >> 6;
        const uint32_t n8 = wg.colstart[64 * t + 64] - wg.colstart[64 * t];
        const uint32_t tx = t % g.tiles_x, ty = t / g.tiles_x;
        const float cf = static_cast<float>(g.c);
        const float area = static_cast<float>(min(8u, g.gx - 8 * tx)) *
                           static_cast<float>(min(8u, g.gy - 8 * ty)) * cf * cf;
        const float per = static_cast<float>(fetch + 1);
        const float r2 = sqrtf(per * area * 0.31830989f / static_cast<float>(max(n8, 1u)));
        const double bx = lane_value(qx, 0), by = lane_value(qy, 0), bz = lane_value(qz, 0);
        const float dx = static_cast<float>(qx - bx), dy = static_cast<float>(qy - by),
                    dz = static_cast<float>(qz - bz);
        const float2 ex = half_extents<LPQ>(pending, dx), ey = half_extents<LPQ>(pending, dy),
                     ez = half_extents<LPQ>(pending, dz);
        const uint64_t vm = __ballot(pending);
        const int half = __popcll(vm & (LPQ == 1 ? 0xFFFFFFFFull : 0xFFFFull));
        const int rest = __popcll((LPQ == 1 ? vm >> 32 : vm >> 16) & (LPQ == 1 ? 0xFFFFFFFFull : 0xFFFFull));
        const float va = half ? ex.x * ey.x * ez.x / static_cast<float>(half) : INFINITY;
        const float vb = rest ? ex.y * ey.y * ez.y / static_cast<float>(rest) : INFINITY;
        const float v = fminf(va, vb);
        const float r3 = v < INFINITY ? cbrtf(per * v * 0.23873241f) : 0.0f;
        const float est = fmaxf(r2, r3);
        r_first = fminf(kRadiusFactor * est, r_cap);
        // Where the estimate itself is beyond the largest radius, nearly every
        // row would be left after all rounds (500k points of a uniform
        // volume, k 32: 1.0 of 8.6 ms): they are left at once.
        if (est > r_cap) {
            defer |= pending;
            pending = false;
        }
    }
    uint64_t cnt_pass = 0, cnt_cand = 0, cnt_sort = 0;
    for (int round = 0; round < (kBail ? 2 : 3); ++round) {
        // The round's group: the pending lanes with as many tries behind them
        // as the first pending one.
        const uint64_t pm = __ballot(pending);
        if (!pm) break;
        const int first = __builtin_ctzll(pm);
        const double bx = lane_value(qx, first), by = lane_value(qy, first),
                     bz = lane_value(qz, first);
        const float rx = static_cast<float>(qx - bx), ry = static_cast<float>(qy - by),
                    rz = static_cast<float>(qz - bz);
        const uint32_t first_tries = lane_u32(tries, first);
        bool act = pending && tries == first_tries;
        float r = r_first;
        StageBox B;
        bool got = false;
        int refine = 0;
        for (int step = 0; step < 16; ++step) {
            const float lx = wave_min_f32(act ? rx : INFINITY), ux = -wave_min_f32(act ? -rx : INFINITY);
            const float ly = wave_min_f32(act ? ry : INFINITY), uy = -wave_min_f32(act ? -ry : INFINITY);
            const float lz = wave_min_f32(act ? rz : INFINITY), uz = -wave_min_f32(act ? -rz : INFINITY);
            const float r_need_max = fminf(-wave_min_f32(act ? -r_need : 0.0f), r_cap);
            r = fmaxf(r, r_need_max);
            // Faces at least r from every active query: the offsets' FP32
            // rounding and the FP64 rounding of the faces taken off.
            const float W = fmaxf(fmaxf(fmaxf(-lx, ux), fmaxf(-ly, uy)), fmaxf(-lz, uz)) + r;
            const double pad = static_cast<double>(r) + 3e-7 * static_cast<double>(W) + wg.margin;
            B.X0 = bx + static_cast<double>(lx) - pad;
            B.X1 = bx + static_cast<double>(ux) + pad;
            B.Y0 = by + static_cast<double>(ly) - pad;
            B.Y1 = by + static_cast<double>(uy) + pad;
            B.Z0 = bz + static_cast<double>(lz) - pad;
            B.Z1 = bz + static_cast<double>(uz) + pad;
            // Grid cells by the points' own rule, so that a point inside the
            // faces is inside the cells.
            const Box b{uniform_i32(static_cast<int>(cell_coord(B.X0, g.ox, g.inv_c, g.gx))),
                        uniform_i32(static_cast<int>(cell_coord(B.X1, g.ox, g.inv_c, g.gx))),
                        uniform_i32(static_cast<int>(cell_coord(B.Y0, g.oy, g.inv_c, g.gy))),
                        uniform_i32(static_cast<int>(cell_coord(B.Y1, g.oy, g.inv_c, g.gy))),
                        uniform_i32(static_cast<int>(cell_coord(B.Z0, g.oz, g.inv_cz, g.gz))),
                        uniform_i32(static_cast<int>(cell_coord(B.Z1, g.oz, g.inv_cz, g.gz)))};
            const uint64_t ncb = static_cast<uint64_t>(b.x1 - b.x0 + 1) *
                                 static_cast<uint64_t>(b.y1 - b.y0 + 1);
            bool over = ncb > kStageCols * 64u;
            if (!over) {
                uint32_t lo[kStageCols], len[kStageCols], part = 0;
                box_columns(a, wg, b, static_cast<int>(ncb), lane, lo, len);
#pragma unroll
                for (int i = 0; i < kStageCols; ++i) part += min(len[i], 1u << 20);
                const uint32_t incl = wave_scan_u32(part);
                const uint32_t N = lane_u32(incl, 63);
                // Where the box turns out denser than the first estimates, the
                // radius its own density asks for.
                if (refine < 2 && r > r_need_max) {
                    const float ex = static_cast<float>(b.x1 - b.x0 + 1) * static_cast<float>(g.c);
                    const float ey = static_cast<float>(b.y1 - b.y0 + 1) * static_cast<float>(g.c);
                    const float ez = static_cast<float>(b.z1 - b.z0 + 1) * static_cast<float>(g.cz);
                    const float per = static_cast<float>(fetch + 1) / static_cast<float>(max(N, 1u));
                    const float r2 = sqrtf(per * ex * ey * 0.31830989f);
                    const float r3 = cbrtf(per * ex * ey * ez * 0.23873241f);
                    const float rn = fmaxf(kRadiusFactor * fmaxf(r2, r3), r_need_max);
                    ++refine;
                    if (rn < 0.85f * r) {
                        r = fmaxf(rn, 0.5f * r);
                        continue;
                    }
                }
                over = N > kStageRaw || N == 0;
                if (!over) {
                    over = !size_box(B, r) ||
                           !stage_points(cv, S, lo, len, incl - part, N, B, lane);
                }
            }
            if (!over) {
                got = true;
                break;
            }
            if (kBail && round == 0) return true;
            // Too many: the half of the group that holds its first query.
            const float dx = ux - lx, dy = uy - ly, dz = uz - lz;
            const float big = fmaxf(dx, fmaxf(dy, dz));
            if (!(big > 0.0f)) break;  // all at one place
            const float v = dx == big ? rx : (dy == big ? ry : rz);
            const float mid = 0.5f * (dx == big ? lx + ux : (dy == big ? ly + uy : lz + uz));
            // (the first query is the base: its offset is 0)
            act = act && (v <= mid) == (0.0f <= mid);
        }
        if (!got) {
            defer |= act;
            pending = pending && !act;
            continue;
        }
        // The lane's cells at radius rl.
        float rl = r;
        const float fx = static_cast<float>(qx - B.X0), fy = static_cast<float>(qy - B.Y0),
                    fz = static_cast<float>(qz - B.Z0);
        // (a hair wider than the radius, so that rounding loses no point)
        const float wider = 1e-6f * (fabsf(fx) + fabsf(fy) + fabsf(fz)) +
                            static_cast<float>(wg.margin);
        CellRange w = stage_range(B, act, fx, fy, fz, r * 1.0001f + wider);
        // Where the box is denser around this query than its radius asks for,
        // a smaller one.
        {
            uint32_t seen = 0;
            for (int z = w.z0; z <= w.z1; ++z)
                for (int y = w.y0; y <= w.y1; ++y) {
                    const int row = (z * B.ny + y) * B.nx;
                    seen += S.cell[row + w.x1 + 1] - S.cell[row + w.x0];
                }
            // At least a quarter of those seen are inside the radius, and
            // their number falls at most with its cube.
            const float in = 0.25f * static_cast<float>(seen);
            const float want = kListFactor * static_cast<float>(fetch + 1);
            if (in > want) {
                rl = fminf(fmaxf(r * cbrtf(want / in), r_need), r);
                w = stage_range(B, act, fx, fy, fz, rl * 1.0001f + wider);
            }
        }
        cnt_pass += static_cast<uint64_t>(__popcll(__ballot(act)));
        // The walk.
        const double E0 = static_cast<double>(rl) * static_cast<double>(rl);
        double E = act ? E0 : -1.0;
        uint32_t cnt = 0, seen = 0;
        bool cut = false;   // entries below E0 may have been left out
        for (int dz = 0; __ballot(w.z0 + dz <= w.z1); ++dz) {
            for (int dy = 0; __ballot(w.y0 + dy <= w.y1); ++dy) {
                uint32_t p = 0, e = 0;
                if (w.y0 + dy <= w.y1 && w.z0 + dz <= w.z1) {
                    const int row = ((w.z0 + dz) * B.ny + w.y0 + dy) * B.nx;
                    p = S.cell[row + w.x0] + part;
                    e = S.cell[row + w.x1 + 1];
                    seen += p < e ? (e - p + LPQ - 1) / LPQ : 0u;
                }
                while (__ballot(p < e)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t t = p < e ? p : 0u;
                        const uint64_t db = dist_bits(qx, qy, qz, S.x[t], S.y[t], S.z[t]);
                        const double d2 = bits_d2(db);
                        my[cnt * 64] = list_key(d2, t);
                        cnt += (p < e && d2 < E) ? 1u : 0u;
                        p += LPQ;
                    }
                    if (__ballot(cnt > CAP - 4)) {
                        uint32_t k[CAP];
                        load_sorted<CAP>(my, cnt, k);
                        cnt_sort += 1;
#pragma unroll
                        for (int i = 0; i < TM; ++i) my[i * 64] = k[i];
                        if (cnt >= keep) {
                            E = fmin(E, key_above(my[(keep - 1) * 64]));
                            cnt = keep;
                            cut = true;
                        }
                    }
                }
            }
        }
        cnt_cand += seen;
        uint32_t idx[TM];
        uint64_t d[TM];
        {
            uint32_t k[CAP];
            load_sorted<CAP>(my, cnt, k);
            cnt_sort += 1;
            if (LPQ == 2) {
                // The TM smallest of the pair's two lists.
                uint32_t m[TM];
#pragma unroll
                for (int i = 0; i < TM; ++i)
                    m[i] = min(k[i], static_cast<uint32_t>(__shfl_xor(static_cast<int>(k[TM - 1 - i]), 32)));
                sort_net<TM>(m);
#pragma unroll
                for (int i = 0; i < TM; ++i) k[i] = m[i];
                cnt += static_cast<uint32_t>(__shfl_xor(static_cast<int>(cnt), 32));
                const int other_cut = __shfl_xor(cut ? 1 : 0, 32);
                cut = cut || other_cut != 0;
            }
            const uint32_t lim = min(cnt, keep);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                my[i * 64] = k[i];
                const bool has = static_cast<uint32_t>(i) < lim;
                const uint32_t t = has ? k[i] & kSlotMask : 0u;
                const uint64_t v = dist_bits(qx, qy, qz, S.x[t], S.y[t], S.z[t]);
                idx[i] = has ? t : kInfU;
                d[i] = has ? v : kInfD;
                if (i % 8 == 7) __builtin_amdgcn_sched_barrier(0);
            }
        }
        // The largest coarse distance put in exact order: no entry cut away
        // has a smaller one.
        cut = cut || cnt >= keep;
        const double last = key_below(my[(keep - 1) * 64]);
        // Exact (d2, id) order: neighbors out of order change places
        // until none is (the coarse order is right but for near-equal
        // distances).
        for (int pass = 0; pass < TM; ++pass) {
            bool any = false;
#pragma unroll
            for (int i = 1; i < TM; ++i) {
                bool sw = d[i] < d[i - 1];
                const bool eq = d[i] == d[i - 1] && d[i] != kInfD;
                if (__ballot(eq)) {
                    if (eq) sw = cv.perm[S.j[idx[i]]] < cv.perm[S.j[idx[i - 1]]];
                }
                const uint64_t u = sw ? d[i] : d[i - 1], v = sw ? d[i - 1] : d[i];
                const uint32_t iu = sw ? idx[i] : idx[i - 1], iv = sw ? idx[i - 1] : idx[i];
                d[i - 1] = u;
                d[i] = v;
                idx[i - 1] = iu;
                idx[i] = iv;
                any |= sw;
            }
            if (!__ballot(any)) break;
        }
        // In (d2, id) order; the list holds slots now.
        uint32_t* list = S.list;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < TM; ++i) list[i * kListRow + lane] = idx[i];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // The fetch-th and (fetch + 1)-th distances.
        auto dist_at = [&](uint32_t i) {
            const uint32_t t = list[i * kListRow + lane];
            return t == kInfU ? kInfD : dist_bits(qx, qy, qz, S.x[t], S.y[t], S.z[t]);
        };
        const uint64_t dk = dist_at(fetch - 1), dn = dist_at(fetch);
        bool tie = dk == dn && dk != kInfD;
        if (wg.stride > 1 || a.mode == 2) {  // equal neighbors anywhere in the list
            tie = false;
#pragma unroll
            for (int i = 1; i < TM; ++i)
                tie |= static_cast<uint32_t>(i) <= fetch && d[i] == d[i - 1] && d[i] != kInfD;
        }
        // (points outside the staged box are farther than rl but for the
        // rounding of one distance)
        const bool in_ball = act && cnt >= fetch && bits_d2(dk) < E0 * (1.0 - 1e-12);
        const bool done = in_ball && (!cut || (dn != kInfD && bits_d2(dn) < last));
        store_rows(a, wg, s, lane, done && part == 0, tie, qx, qy, qz, S.x, S.y, S.z, S.j, list);
        // What is left: a larger radius, or the growing search.
        const bool again = act && !done;
        const bool few = __popcll(__ballot(again && part == 0)) <= kLaneFew;
        if (again) {
            ++tries;
            const float f = sqrtf(1.5f * static_cast<float>(fetch) /
                                  static_cast<float>(max(cnt, 1u)));
            const bool give_up = few || in_ball || rl >= r_cap;
            r_need = rl * fminf(fmaxf(f, 1.3f), 2.0f);
            defer |= give_up;
            pending = !give_up;
        } else if (done) {
            pending = false;
        }
        wave_lds_order();  // the next round stages over this one's box
    }
    // Lanes still pending: their last round failed, or its box was halved
    // without them.
    defer |= pending;
    defer = defer && part == 0;
    const uint64_t dm = __ballot(defer);
    if (dm) {
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(a.out.nflagged + 3, static_cast<uint32_t>(__popcll(dm)));
        at = lane_u32(at, 0) + lanes_below64(dm);
        if (defer) a.out.deferred[at] = static_cast<uint32_t>(s);
    }
    if (a.out.counters) {
        atomicAdd(a.out.counters + 1, static_cast<unsigned long long>(cnt_cand));
        if (lane == 0) {
            atomicAdd(a.out.counters + 0, static_cast<unsigned long long>(cnt_pass));
            atomicAdd(a.out.counters + 2, static_cast<unsigned long long>(cnt_sort));
            atomicAdd(a.out.counters + 3, static_cast<unsigned long long>(nq));
        }
    }
    return false;
}

// One group per wave; groups too heavy for one box are listed in out.heavy.
template <int CAP, int TM, int WPE, bool kTiled>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void k_knn_lane(KnnArgs a)
{
    __shared__ StageShared<CAP> S;
    const uint32_t task = xcd_logical_block(blockIdx.x, gridDim.x);
    WaveGrid wg;
    uint64_t q0;
    int nq;
    if (!wave_queries<kTiled>(a, task, a.q_per_wave, wg, q0, nq)) return;
    if (kTiled && (wg.fetch > a.fetch_hi || wg.fetch < a.fetch_lo)) return;
    if (search_group<CAP, TM, 1, true>(a, wg, q0, nq, S) && __lane_id() == 0)
        a.out.heavy[atomicAdd(a.out.nflagged + 4, 1u)] = task;
}

// The heavy groups, half a group at a time with two lanes per query: half
// the queries need a smaller box, and each walks it in half the steps.  The
// waves draw halves until none is left (their number is read on the device).
template <int CAP, int TM, int WPE, bool kTiled>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void k_knn_pair(KnnArgs a)
{
    __shared__ StageShared<CAP> S;
    const uint32_t halves = 2u * a.out.nflagged[4];
    for (;;) {
        uint32_t h = 0;
        if (__lane_id() == 0) h = atomicAdd(a.out.nflagged + 7, 1u);
        h = lane_u32(h, 0);
        if (h >= halves) return;
        WaveGrid wg;
        uint64_t q0;
        int nq;
        if (!wave_queries<kTiled>(a, a.out.heavy[h >> 1], a.q_per_wave, wg, q0, nq)) continue;
        const int first = 32 * static_cast<int>(h & 1u);
        if (nq <= first) continue;
        search_group<CAP, TM, 2, false>(a, wg, q0 + first, min(nq - first, 32), S);
    }
}

// ------------------------------------------------- wave-per-query search --
//
// Neighborhoods too large for the query-per-lane search (more than
// kLaneMaxFetch entries; its lists and registers grow with them), and those of
// 22 entries and more on small clouds: the
// wave's queries form groups that share a 2 x 2 block of columns and a short
// z range, and one candidate box of up to 256 points held in registers; each
// query's FP64 distances are selected by ballots across the wave.  Rows whose
// box holds too many points, or that it does not certify, go to k_knn_rest;
// but where the latter are most of the wave's and one cloud's launch fills the
// chip the wave searches them itself, from its groups' half-widths on (such
// clouds leave rows everywhere, so the waves stay even; tiles of a batch differ:
// 64 tiles of 20k points, k 16 and 48, 5.4 ms so and 5.0).
//
// Search times, ms, with 16 / 32 / 64 queries per wave: 1M points, k 48, 4.6 /
// 4.8 / 5.1; 60k points, k 48, 0.43 / 0.56 / 0.69; 5k points, k 40, 0.16 / 0.21 /
// 0.35.  Uncertified rows by the waves themselves and by k_knn_rest: 500k points
// of a uniform volume, k 48, 6.1 and 7.1; of normal density, k 40, 4.1 and 4.4;
// 60k points, k 60, where 3750 waves leave the chip half empty, 1.05 and 0.58.
template <bool kTiled>
// Four waves per SIMD: the selection is a chain of ballots and LDS round
// trips, so more resident waves hide more of its latency.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_knn_group(KnnArgs a)
{
    extern __shared__ uint32_t s_lds[];
    const int lane = __lane_id();
    WaveGrid wg;
    uint64_t q0;
    int nq;
    // A task's queries, group_q of them to a wave.
    const uint32_t parts = static_cast<uint32_t>(a.q_per_wave / a.group_q);
    const uint32_t block = xcd_logical_block(blockIdx.x, gridDim.x);
    if (!wave_queries<kTiled>(a, block / parts, a.q_per_wave, wg, q0, nq)) return;
    if (kTiled && (wg.fetch > a.fetch_hi || wg.fetch < a.fetch_lo)) return;
    const int first = static_cast<int>(block % parts) * a.group_q;
    if (nq <= first) return;
    q0 += first;
    nq = min(nq - first, a.group_q);
    const CloudView& cv = a.cv;
    const GridParams& g = wg.g;
    const int fetch = wg.fetch;
    const int k = wg.k;
    // LDS: a 64-entry compaction scratch of 16 bytes per entry, twice, then
    // (features) the queries' neighbor lists.
    uint32_t* scratch = s_lds;
    uint32_t* nbr = s_lds + kScratchWords;
    const uint32_t zmask = (1u << g.bz) - 1u;

    uint8_t my_flags = 0;
    uint64_t left = 0;  // the wave's queries not settled here
    int my_ring = 1;    // the first box of the lane's query if it is left
    uint64_t cnt[3] = {0, 0, 0};  // search passes, candidates, selections
    int qi = 0;
    int rg_prev = 1;  // box half-width of the previous group (density guess)
    // Features with stride 1 keep each neighborhood as a set: the exact-count
    // selection serves them; lists, and strided neighborhoods, need the
    // (d2, id) order.
    const bool as_set = a.mode == 0 && wg.stride == 1;
    // The previous query's threshold, the first one tried (queries in sorted
    // order are close, with similar neighborhood radii).
    double hint = INFINITY;
    // The wave's queries, one per lane, loaded once: coordinates and keys.
    const bool lane_q = lane < nq;
    const double wx = lane_q ? cv.sx[q0 + lane] : 0.0;
    const double wy = lane_q ? cv.sy[q0 + lane] : 0.0;
    const double wz = lane_q ? cv.sz[q0 + lane] : 0.0;
    const uint32_t wkey = lane_q ? cv.keys[q0 + lane] : 0u;
    while (qi < nq) {
        // The group: the run of queries from qi that lie in one 2x2 block of
        // columns (one column if the block is too dense) with z cells within
        // group_z of the first query's.  All of them share one candidate box:
        // the block grown by rg columns on each side, z cells of the members
        // grown by rg.
        const uint64_t s0 = q0 + qi;
        const bool in_range = qi + lane < nq;
        // (shuffled by every lane: a lane outside the wave's queries is still
        // the source of another's key)
        const uint32_t key_sh =
            static_cast<uint32_t>(__shfl(static_cast<int>(wkey), (qi + lane) & 63));
        const uint32_t key_l = in_range ? key_sh : 0u;
        const uint32_t key0 = lane_u32(key_l, 0);
        const int cz0 = static_cast<int>(key0 & zmask);
        const int cz_l = static_cast<int>(key_l & zmask);
        const bool zok = in_range && abs(cz_l - cz0) <= a.tune.group_z;
        const double fx = lane_value(wx, qi), fy = lane_value(wy, qi);
        const int qcx = static_cast<int>(cell_coord(fx, g.ox, g.inv_c, g.gx));
        const int qcy = static_cast<int>(cell_coord(fy, g.oy, g.inv_c, g.gy));
        const uint32_t need = static_cast<uint32_t>(fetch + 1);
        int level = 1;
        int gm = 0, zmin = cz0, zmax = cz0, rg = rg_prev;
        Box box{};
        uint32_t lo = 0, len = 0, tot = 0, excl = 0;
        for (int attempt = 0; attempt < 6; ++attempt) {
            const uint32_t shift = g.bz + 2u * static_cast<uint32_t>(level);
            const bool member = zok && (key_l >> shift) == (key0 >> shift);
            const uint64_t mm = __ballot(member);
            gm = (~mm == 0ull) ? 64 : __builtin_ctzll(~mm);
            int zl = lane < gm ? cz_l : cz0, zh = zl;
#pragma unroll
            for (int m = 32; m > 0; m >>= 1) {
                zl = min(zl, __shfl_xor(zl, m));
                zh = max(zh, __shfl_xor(zh, m));
            }
            zmin = uniform_i32(zl);
            zmax = uniform_i32(zh);
            const int bx0 = level ? (qcx & ~1) : qcx, by0 = level ? (qcy & ~1) : qcy;
            const int bw = level ? 2 : 1;
            box = Box{bx0 - rg, bx0 + bw - 1 + rg, by0 - rg, by0 + bw - 1 + rg, zmin - rg,
                      zmax + rg};
            box_ranges(a, wg, box, 0, lane, static_cast<uint32_t>(a.tune.small_col), lo, len);
            const uint32_t incl = wave_incl_scan_u32(len, lane);
            tot = lane_u32(incl, 63);
            excl = incl - len;
            // Half-width the local density asks for: the need-th neighbor
            // radius of a surface of this 2-D density, with 10% slack.
            const int width = bw + 2 * rg;
            const double area = static_cast<double>(width * width) * g.c * g.c;
            int est = 3;
            if (tot > 0) {
                const double rk = sqrt(static_cast<double>(need) * area /
                                       (3.141592653589793 * static_cast<double>(tot)));
                est = static_cast<int>(ceil(1.1 * rk / g.c));
                // rg <= 3 keeps the box within 64 columns ((2 + 2 rg)^2),
                // the one box_ranges chunk this path reads.
                est = est < 1 ? 1 : (est > 3 ? 3 : est);
            }
            if (tot > kGroupCand) {
                if (rg > 1) {
                    rg = min(rg - 1, est);
                    continue;
                }
                if (level == 1) {
                    level = 0;
                    continue;
                }
                break;  // one dense column: searched query by query
            }
            if (est > rg) {
                rg = est;
                continue;
            }
            break;
        }
        rg_prev = rg;
        const bool cached = tot <= kGroupCand;

        // Shared candidates of the group's box, cached in registers.
        double px[kGroupBatches], py[kGroupBatches], pz[kGroupBatches];
        uint32_t pid[kGroupBatches], pj[kGroupBatches];
#pragma unroll
        for (int b = 0; b < kGroupBatches; ++b) {
            px[b] = py[b] = pz[b] = 0.0;
            pid[b] = pj[b] = kInfU;
            if (cached && static_cast<uint32_t>(b * 64) < tot) {
                const uint32_t t = b * 64 + lane;
                const uint32_t j = candidate_pos(lo, excl, t);
                if (t < tot) {
                    px[b] = cv.sx[j];
                    py[b] = cv.sy[j];
                    pz[b] = cv.sz[j];
                    pid[b] = cv.perm[j];
                    pj[b] = j;
                }
            }
        }

        for (int gi = 0; gi < gm; ++gi) {
            const uint64_t s = s0 + gi;
            const int qslot = qi + gi;
            bool done = false;
            if (cached) {
                const double qx = lane_value(wx, qslot), qy = lane_value(wy, qslot),
                             qz = lane_value(wz, qslot);
                cnt[0] += 1;
                cnt[1] += tot;
                // The candidates' ids and positions are the cache's own.
                uint64_t cd[kGroupBatches];
#pragma unroll
                for (int b = 0; b < kGroupBatches; ++b)
                    cd[b] = (static_cast<uint32_t>(b) * 64u < tot && pj[b] != kInfU)
                                ? dist_bits(qx, qy, qz, px[b], py[b], pz[b])
                                : kInfD;
                const uint32_t nbat = (tot + 63u) >> 6;
                uint64_t E = 0;
                if (as_set && hint < INFINITY && tot >= static_cast<uint32_t>(fetch) &&
                    select_count(cd, nbat, static_cast<uint32_t>(fetch), hint, E)) {
                    // The kept set is {d2 <= E}, with no boundary tie.  It is
                    // certified when its fetch-th distance (<= E) is below
                    // the box clearance less the margin, i.e. when E is, or
                    // when fetch candidates are.
                    cnt[2] += 1;
                    hint = bits_d2(E);
                    const double R = box_clearance(g, box, qx, qy, qz);
                    done = R == INFINITY;
                    if (!done) {
                        const double Rm = R - wg.margin;
                        if (Rm > 0.0) {
                            const double R2 = Rm * Rm;
                            done = bits_d2(E) < R2 ||
                                   count_bits<true>(cd, nbat, d2_bits(R2)) >=
                                       static_cast<uint32_t>(fetch);
                        }
                    }
                    if (done) {
                        // The list in (d2, id) order, as the sorting path
                        // keeps it (so the covariance sums in one order
                        // whatever the grid and launch shape): the kept
                        // entries are compacted into the scratch, and each
                        // of the first fetch lanes counts the entries before
                        // its own and stores its sorted position there.
                        uint32_t base = 0;
#pragma unroll
                        for (int b = 0; b < kGroupBatches; ++b) {
                            if (static_cast<uint32_t>(b) >= nbat) break;
                            const bool kept = cd[b] <= E;
                            const uint64_t m = __ballot(kept);
                            if (kept)
                                reinterpret_cast<uint4*>(scratch)[base + lanes_below64(m)] =
                                    make_uint4(static_cast<uint32_t>(cd[b]),
                                               static_cast<uint32_t>(cd[b] >> 32), pid[b], pj[b]);
                            base += static_cast<uint32_t>(__popcll(m));
                        }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        if (lane < fetch) {
                            const uint4 me = reinterpret_cast<const uint4*>(scratch)[lane];
                            const uint64_t vd = static_cast<uint64_t>(me.x) |
                                                (static_cast<uint64_t>(me.y) << 32);
                            uint32_t rank = 0;
#pragma unroll 4
                            for (int i = 0; i < fetch; ++i)
                                rank += rank_step(reinterpret_cast<const uint4*>(scratch)[i],
                                                  vd, me.z);
                            nbr[qslot * a.lds_stride + rank] = me.w;
                        }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                    }
                } else {
                    // Neighboring queries of a group have similar need-th
                    // distances: the previous one is the first threshold tried.
                    Ent best;
                    select_entries(cd, pid, pj, tot, fetch, lane, scratch, hint, best, cnt);
                    const Ent nth = ent_lane(best, static_cast<int>(min(need, tot)) - 1);
                    hint = nth.d == kInfD ? INFINITY : ent_d2(nth);
                    done = certified(wg, box, ent_lane(best, fetch - 1), qx, qy, qz);
                    if (done) finish_query(a, wg, best, false, s, qslot, lane, nbr, my_flags);
                }
            }
            if (!done) {
                left |= 1ull << qslot;
                if (lane == qslot) my_ring = cached ? rg + 1 : 1;
            }
        }
        qi += gm;
    }
    const uint64_t own = a.group_own ? left & __ballot(my_ring > 1) : 0ull;
    if (2 * __popcll(own) > nq) {
        for (uint64_t m = own; m; m &= m - 1) {
            const int qslot = __builtin_ctzll(m);
            const double qx = lane_value(wx, qslot), qy = lane_value(wy, qslot),
                         qz = lane_value(wz, qslot);
            const int qcx = static_cast<int>(cell_coord(qx, g.ox, g.inv_c, g.gx));
            const int qcy = static_cast<int>(cell_coord(qy, g.oy, g.inv_c, g.gy));
            const int qcz = static_cast<int>(cell_coord(qz, g.oz, g.inv_cz, g.gz));
            Ent best;
            bool incomplete = false;
            search_single(a, wg, qx, qy, qz, qcx, qcy, qcz,
                          min(static_cast<int>(lane_u32(static_cast<uint32_t>(my_ring), qslot)),
                              a.tune.ring_max),
                          lane, scratch, best, incomplete, cnt);
            finish_query(a, wg, best, incomplete, q0 + qslot, qslot, lane, nbr, my_flags);
        }
        left &= ~own;
    }
    if (left) {
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(a.out.nflagged + 3, static_cast<uint32_t>(__popcll(left)));
        at = lane_u32(at, 0) + lanes_below64(left);
        if ((left >> lane) & 1ull) a.out.deferred[at] = static_cast<uint32_t>(q0 + lane);
    }
    if (a.out.counters && lane == 0) {
        atomicAdd(a.out.counters + 0, static_cast<unsigned long long>(cnt[0]));
        atomicAdd(a.out.counters + 1, static_cast<unsigned long long>(cnt[1]));
        atomicAdd(a.out.counters + 2, static_cast<unsigned long long>(cnt[2]));
        atomicAdd(a.out.counters + 3, static_cast<unsigned long long>(nq));
    }
    if (a.mode != 0) return;
    // The lists were written by other lanes of this same wave: order those
    // LDS stores before the loads below (no block barrier: waves of this
    // block may already have exited).
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();

    // One query per lane: FP64 covariance of its neighbor list.
    if (lane >= nq || ((left >> lane) & 1ull)) return;
    const uint64_t s = q0 + lane;
    const uint32_t* list = nbr + lane * a.lds_stride;
    write_cov_record(a, s, k, wx, wy, wz, my_flags, cv.sx, cv.sy, cv.sz,
                     [&](int l) { return list[l]; });
    if (my_flags) {
        const uint32_t slot = atomicAdd(a.out.nflagged, 1u);
        a.out.flagged[slot] = static_cast<uint32_t>(s);
        atomicAdd(a.out.nflagged + ((my_flags & ST_INCOMPLETE) ? 2 : 1), 1u);
    }
}

// The first box of a row's growing search: as many cells to each side as the
// 3 x 3 x 3 cells around it, taken as a sample of a surface and of a volume,
// ask for.
__device__ __forceinline__ int first_ring(const KnnArgs& a, const WaveGrid& wg, int cx, int cy,
                                          int cz, int lane)
{
    const Box b{cx - 1, cx + 1, cy - 1, cy + 1, cz - 1, cz + 1};
    uint32_t lo, len;
    box_ranges(a, wg, b, 0, lane, 0u, lo, len);
    const uint32_t n = lane_u32(wave_incl_scan_u32(len, lane), 63);
    const float c = static_cast<float>(wg.g.c), h = static_cast<float>(wg.g.cz);
    const float per = static_cast<float>(wg.fetch + 1) / static_cast<float>(max(n, 1u));
    const float r = fmaxf(sqrtf(per * 9.0f * c * c * 0.31830989f),
                          cbrtf(per * 27.0f * c * c * h * 0.23873241f));
    const float ring = ceilf(1.1f * r / fminf(c, h));
    return max(a.tune.ring0, min(static_cast<int>(fminf(ring, 1e6f)), min(4, a.tune.ring_max)));
}

// The rows the lane-per-query search left (out.deferred, their count read on
// the device), or every row (tuning "set_select" 0): one wave per row with
// the growing search.  A wave draws a few rows at a time until none is left, so
// that uneven rows spread and the waves at work stay close together in the
// cloud; it holds the lists of kRestHeld rows before one lane each forms their
// covariances.
//
// Bound by the latency of one row's chain of loads and selections, so by the
// waves resident: six per SIMD (80 registers) against four (8 batches of
// candidates instead of 4).  Draws and flagged rows are atomics on one address,
// some 50 ns each, hence more rows per draw when there are many.  Search times
// with four waves, rows of fixed strides and covariances after every four, and
// as it is now, ms: 500k points with strays far off (every row here), k 16, 160
// and 94; 60 dense balls, k 16, 10.4 and 6.8; 4M points, k 48, 24.3 and 18.4.
constexpr uint32_t kRestRows = 4;
constexpr uint32_t kRestRowsMany = 8;
constexpr uint32_t kRestMany = 131072;
constexpr int kRestHeld = 16;
constexpr uint32_t kRestWaves = 8192;

template <bool kTiled>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_knn_rest(KnnArgs a)
{
    extern __shared__ uint32_t s_lds[];
    const int lane = __lane_id();
    uint32_t* scratch = s_lds;
    uint32_t* nbr = s_lds + kScratchWords;
    const uint32_t total = a.all_rows ? static_cast<uint32_t>(a.cv.n) : a.out.nflagged[3];
    const uint32_t per = total >= kRestMany ? kRestRowsMany : kRestRows;
    // Each wave's first rows are its own; the rest are drawn.
    const uint32_t drawn0 = gridDim.x * per;
    uint32_t base = blockIdx.x * per;
    if (base >= total) return;
    uint64_t cnt[3] = {0, 0, 0};  // search passes, candidates, selections
    // The rows held: row p's list at nbr + p * lds_stride, its position, size
    // and flags in lane p.
    int held = 0;
    uint8_t my_flags = 0;
    uint32_t my_s = 0;
    int my_k = 0;
    for (;;) {
        const int nq = base >= total ? 0 : static_cast<int>(min(total - base, per));
        for (int p = 0; p < nq; ++p) {
            const uint32_t s = a.all_rows ? base + p : a.out.deferred[base + p];
            WaveGrid wg;
            if (kTiled) {
                const TileInfo& ti = a.tiles[tile_of(a.starts, a.ntiles, s)];
                if (ti.all_exact) continue;
                tile_grid(a, ti, wg);
            } else {
                cloud_grid(a, wg);
            }
            const GridParams& g = wg.g;
            const double qx = a.cv.sx[s], qy = a.cv.sy[s], qz = a.cv.sz[s];
            const int qcx = uniform_i32(static_cast<int>(cell_coord(qx, g.ox, g.inv_c, g.gx)));
            const int qcy = uniform_i32(static_cast<int>(cell_coord(qy, g.oy, g.inv_c, g.gy)));
            const int qcz = uniform_i32(static_cast<int>(cell_coord(qz, g.oz, g.inv_cz, g.gz)));
            Ent best;
            bool incomplete = false;
            // (what k_knn_group leaves is mostly too dense for it: one ring
            // first; 500k points of normal density, k 40, 4.1 ms against 5.0)
            const int ring = wg.fetch > kLaneMaxFetch ? a.tune.ring0
                                                      : first_ring(a, wg, qcx, qcy, qcz, lane);
            search_single(a, wg, qx, qy, qz, qcx, qcy, qcz, ring, lane, scratch, best, incomplete,
                          cnt);
            finish_query(a, wg, best, incomplete, s, held + p, lane, nbr, my_flags);
            if (lane == held + p) {
                my_s = s;
                my_k = wg.k;
            }
        }
        if (a.mode == 0) held += nq;
        const bool last = nq == 0;
        if (a.mode == 0 && (last || held + static_cast<int>(per) > kRestHeld)) {
            // The lists were written by other lanes of this same wave.
            wave_lds_order();
            if (lane < held && my_k > 0) {
                const uint32_t* list = nbr + lane * a.lds_stride;
                write_cov_record(a, my_s, my_k, a.cv.sx[my_s], a.cv.sy[my_s], a.cv.sz[my_s],
                                 my_flags, a.cv.sx, a.cv.sy, a.cv.sz,
                                 [&](int l) { return list[l]; });
                if (my_flags) {
                    const uint32_t slot = atomicAdd(a.out.nflagged, 1u);
                    a.out.flagged[slot] = my_s;
                    atomicAdd(a.out.nflagged + ((my_flags & ST_INCOMPLETE) ? 2 : 1), 1u);
                }
            }
            wave_lds_order();
            held = 0;
            my_k = 0;
            my_flags = 0;
        }
        if (last) break;
        base = total;
        if (drawn0 < total) {
            uint32_t d = 0;
            if (lane == 0) d = atomicAdd(a.out.nflagged + 5, per);
            base = drawn0 + lane_u32(d, 0);
        }
    }
    if (a.out.counters && lane == 0) {
        atomicAdd(a.out.counters + 0, static_cast<unsigned long long>(cnt[0]));
        atomicAdd(a.out.counters + 1, static_cast<unsigned long long>(cnt[1]));
        atomicAdd(a.out.counters + 2, static_cast<unsigned long long>(cnt[2]));
    }
}

// ---------------------------------------------------------------------------
// Radius neighborhoods (the stages' `radius` option; KD3Index::radius,
// pdal/private/KDImpl.hpp:398-415, nanoflann radiusSearch): every point whose
// FP64 squared distance (KD3Index's operation order) is strictly below r*r.
// The set is decided by that comparison alone -- no boundary tie, no exact
// re-solve.  A wave takes 64 spatially compact queries, one per lane, and
// stages the points of their bounding box grown by r in LDS, sorted into
// cells, as the kNN search does; each lane walks the runs of cells within r of
// its query, once for the count and the mean (coordinates relative to the
// query) and once more for the FP64 covariance about it.  A group whose box
// holds too many points is halved along its longest axis; where kRadiusFew
// queries still do not fit, the wave's remaining rows go to k_radius_rest, one
// wave per row, which streams the row's columns from memory, 256 candidates at
// a time.
//
// Bound by LDS reads and FP64 instructions.  With one row at a time per
// wavefront, candidates masked by ballots and every covariance entry summed
// across the wave, 1M points of 28 neighbors (median; 5% above 300) took 7.8
// ms; now 1.8 ms.
// kRadiusFew: the search there takes 2.1 ms at 8, 1.88 at 16, 1.81 at 24, 1.78
// at 33, 1.81 without halving: each halving is one more staging round of a
// wave, with fewer lanes at work.
constexpr int kRadiusFew = 32;

struct RadiusArgs {
    CloudView cv;
    double r2;          // r * r, the strict bound on d2
    float r;            // r, rounded up
    double margin;      // of the cells' faces
    int32_t rx, rz;     // box growth in columns and z cells
    int32_t mode;       // 0: covariance records; 1: counts only
    double* cov;        // mode 0: records in sorted order (count in word 7)
    uint32_t* counts;   // mode 1: counts in original order
    uint32_t* rest;     // rows left to k_radius_rest: their number, then they
};

// Candidates of one chunk: d2 bits per register batch (kInfD outside r).
__device__ __forceinline__ void radius_pass1(const double (&px)[kRadBatches],
                                             const double (&py)[kRadBatches],
                                             const double (&pz)[kRadBatches],
                                             const uint32_t (&pj)[kRadBatches], uint32_t n1,
                                             double qx, double qy, double qz, double r2,
                                             uint32_t& cnt, double& sx, double& sy, double& sz)
{
#pragma unroll
    for (int b = 0; b < kRadBatches; ++b) {
        if (static_cast<uint32_t>(b) * 64u >= n1) break;
        const bool valid = pj[b] != kInfU;
        const double d2 = bits_d2(dist_bits(qx, qy, qz, px[b], py[b], pz[b]));
        const bool in = valid && d2 < r2;
        cnt += static_cast<uint32_t>(__popcll(__ballot(in)));
        if (in) {
            sx += px[b] - qx;
            sy += py[b] - qy;
            sz += pz[b] - qz;
        }
    }
}

__device__ __forceinline__ void radius_pass2(const double (&px)[kRadBatches],
                                             const double (&py)[kRadBatches],
                                             const double (&pz)[kRadBatches],
                                             const uint32_t (&pj)[kRadBatches], uint32_t n1,
                                             double qx, double qy, double qz, double r2,
                                             double mx, double my, double mz, double (&c)[6])
{
#pragma unroll
    for (int b = 0; b < kRadBatches; ++b) {
        if (static_cast<uint32_t>(b) * 64u >= n1) break;
        const bool valid = pj[b] != kInfU;
        const double d2 = bits_d2(dist_bits(qx, qy, qz, px[b], py[b], pz[b]));
        if (valid && d2 < r2) {
            const double dx = (px[b] - qx) - mx, dy = (py[b] - qy) - my, dz = (pz[b] - qz) - mz;
            c[0] += dx * dx;
            c[1] += dx * dy;
            c[2] += dx * dz;
            c[3] += dy * dy;
            c[4] += dy * dz;
            c[5] += dz * dz;
        }
    }
}

struct RadiusShared {
    static constexpr bool kPositions = false;
    double x[kStageMax], y[kStageMax], z[kStageMax];
    uint32_t j[1];
    uint32_t cell[kStageCells + 2];
    uint32_t pos[kStageRaw];
};

__device__ __forceinline__ void write_radius_row(const RadiusArgs& a, uint64_t s, uint32_t cnt,
                                                 const double (&c)[6])
{
    if (a.mode == 1) {
        a.counts[a.cv.perm[s]] = cnt;
        return;
    }
    const double den = static_cast<double>(cnt) - 1.0;
    double* rec = a.cov + kCovRecord * s;
#pragma unroll
    for (int i = 0; i < 6; ++i) rec[i] = c[i] / den;
    reinterpret_cast<uint64_t*>(rec)[6] = 0;
    reinterpret_cast<uint64_t*>(rec)[7] = cnt;
}

// One row by the whole wave, streamed from memory.
__device__ __forceinline__ void radius_row(const RadiusArgs& a, const KnnArgs& ka,
                                           const WaveGrid& wg, uint64_t s, int lane)
{
    const CloudView& cv = a.cv;
    const GridParams& g = cv.g;
    const double qx = cv.sx[s], qy = cv.sy[s], qz = cv.sz[s];
    const int qcx = uniform_i32(static_cast<int>(cell_coord(qx, g.ox, g.inv_c, g.gx)));
    const int qcy = uniform_i32(static_cast<int>(cell_coord(qy, g.oy, g.inv_c, g.gy)));
    const int qcz = static_cast<int>(uniform_u32(cv.keys[s]) & ((1u << g.bz) - 1u));
    const Box box{qcx - a.rx, qcx + a.rx, qcy - a.rx, qcy + a.rx, qcz - a.rz, qcz + a.rz};
    const int ncb = (1 + 2 * a.rx) * (1 + 2 * a.rx);
    uint32_t cnt = 0;
    double sx = 0.0, sy = 0.0, sz = 0.0;
    double c[6] = {0, 0, 0, 0, 0, 0};
    for (int pass = 0; pass < (a.mode == 0 ? 2 : 1); ++pass) {
        double mx = 0.0, my = 0.0, mz = 0.0;
        if (pass == 1) {
            const double nn = static_cast<double>(cnt);
            mx = wave_sum_f64(sx) / nn;
            my = wave_sum_f64(sy) / nn;
            mz = wave_sum_f64(sz) / nn;
        }
        // Chunks of 64 columns and 256 candidates.
        for (int cb = 0; cb < ncb; cb += kWave) {
            uint32_t lo, len;
            box_ranges(ka, wg, box, cb, lane, 0u, lo, len);
            const uint32_t incl = wave_incl_scan_u32(len, lane);
            const uint32_t ctot = lane_u32(incl, 63);
            const uint32_t excl = incl - len;
            for (uint32_t t0 = 0; t0 < ctot; t0 += kRadCand) {
                double cx[kRadBatches], cy[kRadBatches], czv[kRadBatches];
                uint32_t cj[kRadBatches];
                const uint32_t n1 = min(ctot - t0, kRadCand);
#pragma unroll
                for (int b = 0; b < kRadBatches; ++b) {
                    cx[b] = cy[b] = czv[b] = 0.0;
                    cj[b] = kInfU;
                    if (static_cast<uint32_t>(b * 64) < n1) {
                        const uint32_t t = t0 + b * 64 + lane;
                        const uint32_t j = candidate_pos(lo, excl, t);
                        if (t < ctot) {
                            cx[b] = cv.sx[j];
                            cy[b] = cv.sy[j];
                            czv[b] = cv.sz[j];
                            cj[b] = j;
                        }
                    }
                }
                if (pass == 0)
                    radius_pass1(cx, cy, czv, cj, n1, qx, qy, qz, a.r2, cnt, sx, sy, sz);
                else
                    radius_pass2(cx, cy, czv, cj, n1, qx, qy, qz, a.r2, mx, my, mz, c);
            }
        }
    }
    if (a.mode == 0) {
#pragma unroll
        for (int i = 0; i < 6; ++i) c[i] = wave_sum_f64(c[i]);
    }
    if (lane == 0) write_radius_row(a, s, cnt, c);
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_radius(RadiusArgs a)
{
    __shared__ RadiusShared S;
    const int lane = __lane_id();
    const CloudView& cv = a.cv;
    const GridParams& g = cv.g;
    const uint64_t q0 = static_cast<uint64_t>(xcd_logical_block(blockIdx.x, gridDim.x)) * 64u;
    if (q0 >= cv.n) return;
    const int nq = static_cast<int>(cv.n - q0 < 64 ? cv.n - q0 : 64);
    // box_ranges and box_columns read only these fields of the kNN arguments.
    KnnArgs ka{};
    ka.cv = cv;
    WaveGrid wg{};
    wg.g = g;
    wg.colstart = cv.colstart;
    const bool valid = lane < nq;
    const uint64_t s = valid ? cv.qord[q0 + lane] : q0;
    const double qx = valid ? cv.sx[s] : 0.0;
    const double qy = valid ? cv.sy[s] : 0.0;
    const double qz = valid ? cv.sz[s] : 0.0;
    const float r = a.r;
    bool pending = valid && stage_takes_point(qx, qy, qz) && r < 1e18f && r > 1e-18f;
    uint64_t left = __ballot(valid && !pending);  // rows for k_radius_rest
    for (;;) {
        const uint64_t pm = __ballot(pending);
        if (!pm) break;
        const int first = __builtin_ctzll(pm);
        const double bx = lane_value(qx, first), by = lane_value(qy, first),
                     bz = lane_value(qz, first);
        const float rx = static_cast<float>(qx - bx), ry = static_cast<float>(qy - by),
                    rz = static_cast<float>(qz - bz);
        bool act = pending;
        bool got = false;
        StageBox B;
        for (;;) {
            const float lx = wave_min_f32(act ? rx : INFINITY), ux = -wave_min_f32(act ? -rx : INFINITY);
            const float ly = wave_min_f32(act ? ry : INFINITY), uy = -wave_min_f32(act ? -ry : INFINITY);
            const float lz = wave_min_f32(act ? rz : INFINITY), uz = -wave_min_f32(act ? -rz : INFINITY);
            // Faces at least r from every active query: the offsets' FP32
            // rounding and the FP64 rounding of the faces taken off.
            const float W = fmaxf(fmaxf(fmaxf(-lx, ux), fmaxf(-ly, uy)), fmaxf(-lz, uz)) + r;
            const double pad = static_cast<double>(r) + 3e-7 * static_cast<double>(W) + a.margin;
            B.X0 = bx + static_cast<double>(lx) - pad;
            B.X1 = bx + static_cast<double>(ux) + pad;
            B.Y0 = by + static_cast<double>(ly) - pad;
            B.Y1 = by + static_cast<double>(uy) + pad;
            B.Z0 = bz + static_cast<double>(lz) - pad;
            B.Z1 = bz + static_cast<double>(uz) + pad;
            // Grid cells by the points' own rule, so that a point inside the
            // faces is inside the cells.
            const Box b{uniform_i32(static_cast<int>(cell_coord(B.X0, g.ox, g.inv_c, g.gx))),
                        uniform_i32(static_cast<int>(cell_coord(B.X1, g.ox, g.inv_c, g.gx))),
                        uniform_i32(static_cast<int>(cell_coord(B.Y0, g.oy, g.inv_c, g.gy))),
                        uniform_i32(static_cast<int>(cell_coord(B.Y1, g.oy, g.inv_c, g.gy))),
                        uniform_i32(static_cast<int>(cell_coord(B.Z0, g.oz, g.inv_cz, g.gz))),
                        uniform_i32(static_cast<int>(cell_coord(B.Z1, g.oz, g.inv_cz, g.gz)))};
            const uint64_t ncb = static_cast<uint64_t>(b.x1 - b.x0 + 1) *
                                 static_cast<uint64_t>(b.y1 - b.y0 + 1);
            if (ncb <= kStageCols * 64u) {
                uint32_t lo[kStageCols], len[kStageCols], part = 0;
                box_columns(ka, wg, b, static_cast<int>(ncb), lane, lo, len);
#pragma unroll
                for (int i = 0; i < kStageCols; ++i) part += min(len[i], 1u << 20);
                const uint32_t incl = wave_scan_u32(part);
                const uint32_t N = lane_u32(incl, 63);
                if (N <= kStageRaw) {
                    got = size_box(B, r) &&
                          stage_points(cv, S, lo, len, incl - part, N, B, lane);
                }
            }
            if (got) break;
            const float dx = ux - lx, dy = uy - ly, dz = uz - lz;
            const float big = fmaxf(dx, fmaxf(dy, dz));
            const uint64_t am = __ballot(act);
            if (!(big > 0.0f) || __popcll(am) <= kRadiusFew) break;
            // Too many: the half of the group that holds its first query.
            const float v = dx == big ? rx : (dy == big ? ry : rz);
            const float mid = 0.5f * (dx == big ? lx + ux : (dy == big ? ly + uy : lz + uz));
            // (the first query is the base: its offset is 0)
            const bool keep = act && (v <= mid) == (0.0f <= mid);
            if (__ballot(keep) == am) break;  // the extent is within rounding
            act = keep;
        }
        if (!got) {  // the rest of the wave is as dense
            left |= __ballot(pending);
            break;
        }
        // The lane's cells, a hair wider than r, so that rounding loses no
        // point.
        const float fx = static_cast<float>(qx - B.X0), fy = static_cast<float>(qy - B.Y0),
                    fz = static_cast<float>(qz - B.Z0);
        const float e = r * 1.0001f + 1e-6f * (fabsf(fx) + fabsf(fy) + fabsf(fz)) +
                        static_cast<float>(a.margin);
        const CellRange w = stage_range(B, act, fx, fy, fz, e);
        const double r2 = act ? a.r2 : -1.0;
        auto walk = [&](auto&& take) {
            for (int dz = 0; __ballot(w.z0 + dz <= w.z1); ++dz)
                for (int dy = 0; __ballot(w.y0 + dy <= w.y1); ++dy) {
                    uint32_t p = 0, end = 0;
                    if (w.y0 + dy <= w.y1 && w.z0 + dz <= w.z1) {
                        const int row = ((w.z0 + dz) * B.ny + w.y0 + dy) * B.nx;
                        p = S.cell[row + w.x0];
                        end = S.cell[row + w.x1 + 1];
                    }
                    while (__ballot(p < end)) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint32_t t = p < end ? p : 0u;
                            // (px - qx: the negative of KD3Index's difference,
                            // with the same square)
                            const double px = S.x[t] - qx, py = S.y[t] - qy, pz = S.z[t] - qz;
                            double d2 = px * px;
                            d2 = d2 + py * py;
                            d2 = d2 + pz * pz;
                            take(px, py, pz, p < end && d2 < r2);
                            ++p;
                        }
                    }
                }
        };
        uint32_t cnt = 0;
        double sx = 0.0, sy = 0.0, sz = 0.0;
        double c[6] = {0, 0, 0, 0, 0, 0};
        if (a.mode == 1) {
            walk([&](double, double, double, bool in) { cnt += in ? 1u : 0u; });
        } else {
            walk([&](double px, double py, double pz, bool in) {
                cnt += in ? 1u : 0u;
                sx += in ? px : 0.0;
                sy += in ? py : 0.0;
                sz += in ? pz : 0.0;
            });
            const double nn = static_cast<double>(cnt);
            const double mx = sx / nn, my = sy / nn, mz = sz / nn;
            walk([&](double px, double py, double pz, bool in) {
                const double dx = in ? px - mx : 0.0, dy = in ? py - my : 0.0,
                             dz = in ? pz - mz : 0.0;
                c[0] += dx * dx;
                c[1] += dx * dy;
                c[2] += dx * dz;
                c[3] += dy * dy;
                c[4] += dy * dz;
                c[5] += dz * dz;
            });
        }
        if (act) write_radius_row(a, s, cnt, c);
        pending = pending && !act;
        wave_lds_order();
    }
    if (left) {
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(a.rest, static_cast<uint32_t>(__popcll(left)));
        at = lane_u32(at, 0) + lanes_below64(left);
        if ((left >> lane) & 1ull) a.rest[1 + at] = static_cast<uint32_t>(s);
    }
}

// The rows k_radius left, their number read on the device.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_radius_rest(RadiusArgs a)
{
    KnnArgs ka{};
    ka.cv = a.cv;
    WaveGrid wg{};
    wg.g = a.cv.g;
    wg.colstart = a.cv.colstart;
    const uint32_t total = a.rest[0];
    for (uint32_t i = blockIdx.x; i < total; i += gridDim.x)
        radius_row(a, ka, wg, uniform_u32(a.rest[1 + i]), __lane_id());
}

// Per sorted row: eigensystem of the stored covariance and every requested
// stage column, written at the row's original index.
// One thread per row: by original id (kFeaturesAll, kFeaturesUnflagged: a
// row whose record carries a search flag is skipped), or the i-th row of
// out.flagged by sorted position (kFeaturesFlagged).

__device__ __forceinline__ void features_row(uint64_t i, const double* __restrict__ cov,
                                             const uint32_t* __restrict__ inv,
                                             const uint32_t* __restrict__ perm, int rows,
                                             const FusedProgram& prog, const KnnOutputs& out,
                                             const TileInfo* __restrict__ tiles,
                                             const uint64_t* __restrict__ starts,
                                             uint32_t ntiles)
{
    uint64_t qid = i, s;
    if (rows == kFeaturesFlagged) {
        s = out.flagged[i];
        qid = perm[s];
    } else {
        s = inv[qid];  // the row's sorted position: one record read
    }
    // The neighborhood size: the row's own count in radius mode, else its
    // tile's k (stages are the same in every tile).
    const double* rec = cov + kCovRecord * s;
    const int k = prog.radius > 0.0
                      ? static_cast<int>(reinterpret_cast<const uint64_t*>(rec)[7])
                      : (tiles ? tiles[tile_of(starts, ntiles, s)].prog.k : prog.k);
    double c[6];
    for (int i = 0; i < 6; ++i) c[i] = rec[i];
    const uint8_t f = static_cast<uint8_t>(reinterpret_cast<const uint64_t*>(rec)[6]);
    if (rows == kFeaturesUnflagged && f) return;  // written after its exact re-solve
    const bool zero = cov_is_zero(c);
    double ev[3] = {0, 0, 0}, vec[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int info = 0;
    // estimaterank has no isZero skip: it takes the singular values of any
    // covariance.
    bool rank_stage = false;
    for (int si = 0; si < prog.nstages; ++si) rank_stage |= prog.st[si].stage == STAGE_RANK;
    if (!zero || rank_stage) info = eigen_sym3(c, ev, vec);
    for (int si = 0; si < prog.nstages; ++si) {
        const StageProgram& sp = prog.st[si];
        double vals[10];
        // Radius mode: covariancefeatures and eigenvalues skip rows with
        // fewer than min_k neighbors (CovarianceFeaturesFilter.cpp:216-223,
        // EigenvaluesFilter.cpp:125-135); normal skips fewer than three.
        uint8_t st = (prog.radius > 0.0 && sp.stage != STAGE_NORMAL && k < prog.min_k)
                         ? static_cast<uint8_t>(ST_FEW_NEIGHBORS)
                         : stage_outputs(sp, k, c, zero, info, ev, vec, vals);
        if (st == 0)
            for (int cc = 0; cc < sp.ncols; ++cc) out.col[sp.col_offset + cc][qid] = vals[cc];
        out.status[si][qid] = st | (f & kReportedSearchFlags);
    }
}

__global__ __launch_bounds__(256) void k_features(const double* __restrict__ cov,
                                                  const uint32_t* __restrict__ inv,
                                                  const uint32_t* __restrict__ perm,
                                                  uint64_t n, int rows, FusedProgram prog,
                                                  KnnOutputs out, const TileInfo* __restrict__ tiles,
                                                  const uint64_t* __restrict__ starts,
                                                  uint32_t ntiles)
{
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    features_row(i, cov, inv, perm, rows, prog, out, tiles, starts, ntiles);
}

// The flagged rows, their count read on the device (a launch whose shape
// does not depend on it, as a captured graph needs).
__global__ __launch_bounds__(256) void k_features_flagged(const double* __restrict__ cov,
                                                          const uint32_t* __restrict__ inv,
                                                          const uint32_t* __restrict__ perm,
                                                          FusedProgram prog, KnnOutputs out,
                                                          const TileInfo* __restrict__ tiles,
                                                          const uint64_t* __restrict__ starts,
                                                          uint32_t ntiles)
{
    const uint64_t n = *out.nflagged;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
        features_row(i, cov, inv, perm, kFeaturesFlagged, prog, out, tiles, starts, ntiles);
}

__global__ __launch_bounds__(256) void k_eigen_batch(const double* __restrict__ cov,
                                                     uint64_t m, double* __restrict__ ev,
                                                     double* __restrict__ vec,
                                                     int32_t* __restrict__ info)
{
    uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= m) return;
    const double* a = cov + 9 * i;
    double c[6] = {a[0], a[3], a[6], a[4], a[7], a[8]};
    double e[3], v[9];
    info[i] = eigen_sym3(c, e, v);
    for (int t = 0; t < 3; ++t) ev[3 * i + t] = e[t];
    for (int t = 0; t < 9; ++t) vec[9 * i + t] = v[t];
}

} // namespace

// The search kernels that serve a result capacity.  List entries and kept
// entries of the query-per-lane instances follow it, and with them LDS and
// registers: 150, 222 and, at 37 entries, already more than the 256 that are left
// (42 to 90 spilled).  Above kLaneMaxFetch the wave-per-query search serves.  So
// it does for 22 entries and more on clouds (or batches) of fewer than kWideMin
// points: the largest instance's waves, 64 queries each, are few and long there.  Search, ms, by that instance and wave per query: 3k
// points in dense balls, k 36, 0.50 and 0.20; 60k airborne points, k 31, 0.62
// and 0.34; 125k, k 36, 0.80 and 0.59.  At 131,072 points the exact tree is built
// beside the search, and finds fewer free slots beside the wave-per-query
// kernel: 200k, k 36, search 1.28 and 0.94, but the call 1.90 and 2.05.
constexpr int kGroupQueries = 16;           // k_knn_group's queries per wave
constexpr uint32_t kGroupMaxTasks = 1u << 24;  // tasks of 64 queries cut into waves of 16
constexpr uint64_t kWideMin = 131072;
static_assert(uint64_t{kGroupMaxTasks} * (kQueriesPerWave / kGroupQueries) * 64 <= 1ull << 32);
constexpr uint32_t kGroupOwnWaves = 16384;  // four rounds of the waves that fit the chip

static int lane_class(int fetch)
{
    return fetch <= 9 ? 0 : fetch <= 21 ? 1 : fetch <= kLaneMaxFetch ? 2 : 3;
}

uint32_t knn_class_bit(int fetch) { return 1u << lane_class(fetch); }

template <bool kTiled>
static void launch_lane(KnnArgs& a, uint32_t classes, uint32_t blocks, hipStream_t s)
{
    int group_lo = kLaneMaxFetch + 1;
    if (a.cv.n < kWideMin && (classes & 4u)) {
        classes = (classes & ~4u) | 8u;
        group_lo = 22;
    }
    bool again = false;
    auto one = [&](uint32_t bit, int lo, int hi, auto lane, auto pair) {
        if (!(classes & bit)) return;
        if (again) {  // the heavy list starts over with each class
            launch_fill_u32(a.out.nflagged + 4, 1, 0u, s);
            launch_fill_u32(a.out.nflagged + 7, 1, 0u, s);
        }
        again = true;
        a.fetch_lo = lo;
        a.fetch_hi = hi;
        hipLaunchKernelGGL(lane, dim3(blocks), dim3(64), 0, s, a);
        hipLaunchKernelGGL(pair, dim3(std::min<uint32_t>(2 * blocks, 2048)), dim3(64), 0, s, a);
    };
    one(1u, 0, 9, k_knn_lane<24, 12, 2, kTiled>, k_knn_pair<20, 12, 2, kTiled>);
    one(2u, 10, 21, k_knn_lane<40, 24, 2, kTiled>, k_knn_pair<32, 24, 2, kTiled>);
    one(4u, 22, kLaneMaxFetch, k_knn_lane<56, 40, 2, kTiled>, k_knn_pair<48, 40, 2, kTiled>);
    if (classes & 8u) {
        // (a launch holds fewer than 2^32 threads)
        if (blocks >= kGroupMaxTasks) a.group_q = a.q_per_wave;
        a.fetch_lo = group_lo;
        a.fetch_hi = kMaxFetch - 1;
        const size_t lds = (kScratchWords + (a.mode != 0 ? 0 : a.group_q * a.lds_stride)) *
                           sizeof(uint32_t);
        const uint32_t waves = blocks * static_cast<uint32_t>(a.q_per_wave / a.group_q);
        a.group_own = !kTiled && waves >= kGroupOwnWaves;
        hipLaunchKernelGGL(k_knn_group<kTiled>, dim3(waves), dim3(64), lds, s, a);
    }
}

void launch_knn(const CloudView& cv, const FusedProgram& prog, int mode,
                const KnnOutputs& out, const KnnTuning& tune, hipStream_t s,
                const TileTables* tt)
{
    if (cv.n == 0) return;
    KnnArgs a{};
    a.cv = cv;
    a.prog = prog;
    a.out = out;
    a.tune = tune;
    a.mode = mode;
    a.all_rows = tune.set_select ? 0 : 1;
    const int max_k = tt ? tt->max_k : prog.k;
    a.q_per_wave = tt ? tt->q_per_wave
                      : (tune.q_per_wave > 0 ? tune.q_per_wave : kQueriesPerWave);
    a.group_q = tune.q_per_wave > 0 ? a.q_per_wave : kGroupQueries;
    a.lds_stride = max_k | 1;  // odd stride: lanes hit distinct LDS banks
    const GridParams& g = cv.g;
    a.margin = 1e-6 * fmin(g.c, g.cz) +
               1e-15 * (fabs(g.ox) + fabs(g.oy) + fabs(g.oz)) + 1e-300;
    // The rest: a grid for the few rows usually left (the waves draw what more
    // there are).
    const uint32_t rest = static_cast<uint32_t>(
        std::min<uint64_t>(div_up(cv.n, kRestRows), kRestWaves));
    const size_t lds = (kScratchWords + (mode != 0 ? 0 : kRestHeld * a.lds_stride)) *
                       sizeof(uint32_t);
    if (tt) {
        if (!tt->ntasks) return;
        a.tiles = tt->tiles;
        a.starts = tt->starts;
        a.task0 = tt->task0;
        a.ntasks = tt->ntasks;
        a.ntiles = tt->ntiles;
        if (!a.all_rows) launch_lane<true>(a, tt->classes, tt->ntasks, s);
        hipLaunchKernelGGL(k_knn_rest<true>, dim3(rest), dim3(64), lds, s, a);
        return;
    }
    if (!a.all_rows)
        launch_lane<false>(a, knn_class_bit(prog.fetch), div_up(cv.n, a.q_per_wave), s);
    hipLaunchKernelGGL(k_knn_rest<false>, dim3(rest), dim3(64), lds, s, a);
}

void launch_radius(const CloudView& cv, double radius, int mode, double* cov, uint32_t* counts,
                   uint32_t* rest, hipStream_t s)
{
    if (cv.n == 0) return;
    RadiusArgs a{};
    a.cv = cv;
    a.r2 = radius * radius;
    // Every point within r of a query lies within these cells: the cell
    // coordinates' own rounding (relative 4 eps of the grid's span) is
    // covered.
    const GridParams& g = cv.g;
    const double span = fmax(fmax(static_cast<double>(g.gx) * g.c, static_cast<double>(g.gy) * g.c),
                             static_cast<double>(g.gz) * g.cz);
    const double slack = 1e-15 * (span + fabs(g.ox) + fabs(g.oy) + fabs(g.oz));
    a.rx = static_cast<int32_t>(ceil((radius + slack) / g.c));
    a.rz = static_cast<int32_t>(ceil((radius + slack) / g.cz));
    a.r = nextafterf(static_cast<float>(radius), INFINITY);
    a.margin = 1e-6 * fmin(g.c, g.cz) + slack + 1e-300;
    a.mode = mode;
    a.cov = cov;
    a.counts = counts;
    a.rest = rest;
    launch_fill_u32(rest, 1, 0u, s);
    hipLaunchKernelGGL(k_radius, dim3(div_up(cv.n, 64)), dim3(64), 0, s, a);
    const uint32_t blocks = static_cast<uint32_t>(std::min<uint64_t>(cv.n, 8192));
    hipLaunchKernelGGL(k_radius_rest, dim3(blocks), dim3(64), 0, s, a);
}

void launch_features(const CloudView& cv, const FusedProgram& prog,
                     const KnnOutputs& out, const uint32_t* inv, hipStream_t s,
                     const TileTables* tt, int rows, uint64_t nflagged)
{
    const uint64_t n = rows == kFeaturesFlagged ? nflagged : cv.n;
    if (n == 0) return;
    hipLaunchKernelGGL(k_features, dim3(div_up(n, 256)), dim3(256), 0, s, out.cov, inv, cv.perm,
                       n, rows, prog, out, tt ? tt->tiles : nullptr, tt ? tt->starts : nullptr,
                       tt ? tt->ntiles : 0u);
}

void launch_features_flagged(const CloudView& cv, const FusedProgram& prog,
                             const KnnOutputs& out, const uint32_t* inv, uint64_t max_rows,
                             hipStream_t s, const TileTables* tt)
{
    if (!max_rows) return;
    const uint32_t blocks = static_cast<uint32_t>(std::min<uint64_t>(div_up(max_rows, 256), 2048));
    hipLaunchKernelGGL(k_features_flagged, dim3(blocks), dim3(256), 0, s, out.cov, inv, cv.perm,
                       prog, out, tt ? tt->tiles : nullptr, tt ? tt->starts : nullptr,
                       tt ? tt->ntiles : 0u);
}

void launch_eigen_batch(const double* cov, uint64_t m, double* evals,
                        double* evecs, int32_t* info, hipStream_t s)
{
    if (!m) return;
    hipLaunchKernelGGL(k_eigen_batch, dim3(div_up(m, 256)), dim3(256), 0, s, cov, m,
                       evals, evecs, info);
}

} // namespace gf
