// tc_build.hip -- Tree::build on gfx950: bbox, Morton keys, LDS radix sort,
// quadtree topology from sorted keys, upward pass (P2E leaves, E2E parents).
//
// Replaces drivers/sort-sources.cpp:22-132, drivers/upward.cpp:61-314,
// kernels/upward-common.ispc:13-150 and kernels/upward-kernels.m4:18-149.
// Compiled with -ffp-contract=off: keys, centres of mass and radii must be
// rounded exactly as the canonical CPU restatement rounds them, because every
// traversal decision depends on them.
#include "tc_common.h"

#include <cfloat>
#include <climits>
#include <cstring>
#include <type_traits>
#include <vector>

namespace {

// Radix sort of many points: 10-bit digits (three passes over the 30-bit keys;
// with 8-bit digits four), tiles of 1,024 threads with IT keys each.  Few keys per
// thread while the tiles fit the CUs once (a tile's ranking is a chain of LDS round
// trips per key), more where the tiles go in turns: longer digit runs to write, fewer
// tiles to look back over.  Sort of n keys (box, keys, passes), against 8-bit digits
// with tiles of 5,120 keys: 2^16 52.1 -> 48.7 us, 2^20 94.6 -> 89.4, 2^21 146 -> 112,
// 2^22 227 -> 184, 2^23 346 -> 297, 2^24 625 -> 534; with 5 keys per thread 141, 219, 376,
// 750 from 2^21 on, with 8 333 at 2^23 and 652 at 2^24, with 15 126 at 2^21 and 202 at 2^22.
// With the scans on the vector unit and before the look-back: 45.0, 87.5, 110, 179, 291, 522.
constexpr int RS_BITS = 10, RS_BINS = 1 << RS_BITS, RS_PASSES = 3, RS_NT = 1024;
static_assert(RS_PASSES * RS_BITS >= 2 * TC_LMAX, "the passes cover the keys");
constexpr int rs_items(int n) { return n <= 256 * 5 * RS_NT ? 5 : n <= 1 << 22 ? 8 : 15; }
constexpr int SS_BINS = 256;   // one-workgroup sort: 8-bit digits at bits 0, 8, 16, 24
// Key kernel: most workgroups (each adds its digit totals once), and points per
// workgroup and step.  Few points are spread thinner, since a workgroup's
// steps are a chain of memory round trips: 16.9 -> 8 us at 2^16 points, which were 13 steps of 5,120 before.
constexpr int KH_GRID = 1024, KH_TILE_MIN = 1024, KH_TILE_MAX = 5120;
constexpr int SCAN_NT = 1024;  // threads of the census workgroup

__constant__ double c_binom[64 * 64];  // C(n, k) rounded to double, n, k < 64

// ------------------------------------------------------------------ scans
template <int NT>
TC_DEV uint32_t block_scan_excl(uint32_t v, uint32_t *s_w, uint32_t *total)
{
    constexpr int NW = NT / 64;
    const int lane = tc_lane(), wid = threadIdx.x >> 6;
    const uint32_t x = tc_wave_scan(v);
    if (lane == 63)
        s_w[wid] = x;
    __syncthreads();
    if (wid == 0) {
        const uint32_t w = lane < NW ? s_w[lane] : 0u;
        const uint32_t z = tc_wave_scan(w);
        if (lane < NW)
            s_w[lane] = z - w;
        if (lane == NW - 1)
            s_w[NW] = z;
    }
    __syncthreads();
    const uint32_t res = s_w[wid] + x - v;
    if (total)
        *total = s_w[NW];
    __syncthreads();
    return res;
}

__global__ void k_fill_u32(uint32_t *p, uint32_t v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// ------------------------------------------------------------------ sorts of one or two point sets
// One point set of a sort and its device memory.  A solve's sources and targets
// are sorted by the same launches where both are small or middling (a launch
// costs the host about 4 us, a pass of few tiles fills a fraction of the CUs):
// workgroups [0, first set's) take the first set, the rest the second.
struct SortSet {
    const double *x, *y, *v;  // v: sources (Morton keys, records packed); else targets (Hilbert keys)
    double *box;              // {xmin, ymin, ext, scale} out
    uint32_t *keys, *perm;    // out
    uint32_t *k2, *v2;        // scratch of n words each
    double4 *packed;          // source records in input order
    double4 *part;            // bounding-box partials
    uint32_t *bad, *pbad;     // non-finite flag (bit 1: a pass gave up); per-workgroup flags
    uint32_t *lb;             // digit totals, tickets, published counts (lb_words)
    int n, np, ntiles, kgrid, kstep;
};
struct SortSets {
    SortSet s[2];
};

// ------------------------------------------------------------------ bbox
// sort-sources.cpp:44-82 with upward-common.ispc:126-150's accumulators:
// min starts at 1e13, max at 0.  Non-finite coordinates are recorded per
// workgroup in pbad.  Also zeroes the lb words (used after this kernel).
__global__ __launch_bounds__(256) void k_bbox_partial(SortSets sets, int nlb0, int nlb1)
{
    __shared__ double4 s[4];
    const bool second = (int)blockIdx.x >= sets.s[0].np;
    const SortSet &t = second ? sets.s[1] : sets.s[0];
    const int bi = blockIdx.x - (second ? sets.s[0].np : 0), nb = t.np, nlb = second ? nlb1 : nlb0;
    const double *x = t.x, *y = t.y;
    const int n = t.n;
    for (int i = bi * 256 + threadIdx.x; i < nlb; i += nb * 256)
        t.lb[i] = 0u;
    double xmi = 1e13, ymi = 1e13, xma = 0, yma = 0;
    bool nonfinite = false;
    for (int i = bi * 256 + threadIdx.x; i < n; i += nb * 256) {
        const double a = x[i], b = y[i];
        nonfinite |= !isfinite(a) || !isfinite(b);
        xmi = a < xmi ? a : xmi;
        xma = xma < a ? a : xma;
        ymi = b < ymi ? b : ymi;
        yma = yma < b ? b : yma;
    }
    tc_wave_box(xmi, ymi, xma, yma);
    __shared__ uint32_t s_bad;
    if (threadIdx.x == 0)
        s_bad = 0u;
    __syncthreads();
    if (tc_ballot(nonfinite) && tc_lane() == 0)
        s_bad = 1u;
    const int wid = threadIdx.x >> 6;
    if (tc_lane() == 0)
        s[wid] = make_double4(xmi, xma, ymi, yma);
    __syncthreads();
    if (threadIdx.x == 0) {
        double4 r = s[0];
        for (int w = 1; w < 4; ++w) {
            r.x = s[w].x < r.x ? s[w].x : r.x;
            r.y = r.y < s[w].y ? s[w].y : r.y;
            r.z = s[w].z < r.z ? s[w].z : r.z;
            r.w = r.w < s[w].w ? s[w].w : r.w;
        }
        t.part[bi] = r;
        t.pbad[bi] = s_bad;
    }
}

// The box from the partials (one wave): min / max over part[0 .. np), then
// the reference's padded extent.  box[4] = {xmin, ymin, ext, 2^15 / ext}.
TC_DEV void bbox_finish(const double4 *part, int np, double *box)
{
    double xmi = 1e13, xma = 0, ymi = 1e13, yma = 0;
    for (int i = tc_lane(); i < np; i += 64) {
        const double4 r = part[i];
        xmi = r.x < xmi ? r.x : xmi;
        xma = xma < r.y ? r.y : xma;
        ymi = r.z < ymi ? r.z : ymi;
        yma = yma < r.w ? r.w : yma;
    }
    tc_wave_box(xmi, ymi, xma, yma);
    if (tc_lane() == 0) {
        const double ext0 = xma - xmi, ext1 = yma - ymi;
        const double eps = 10000 * DBL_EPSILON;
        double ext = (ext0 < ext1 ? ext1 : ext0) * (1 + 2 * eps);
        if (!(ext > 0))
            ext = 1.0;
        box[0] = xmi - eps * ext;
        box[1] = ymi - eps * ext;
        box[2] = ext;
        box[3] = (1.0 / ext) * (double)(1 << TC_LMAX);
    }
}

// ------------------------------------------------------------------ keys
TC_DEV uint32_t quantise(double v, double vmin, double scale)
{
    double q = floor((v - vmin) * scale);
    if (!(q >= 0))
        q = 0;
    if (q > (double)((1 << TC_LMAX) - 1))
        q = (double)((1 << TC_LMAX) - 1);
    return (uint32_t)q;
}

// Hilbert index of the quantised point (the standard quadrant-rotation
// construction on a 2^15 x 2^15 grid, 30-bit result).  Used to order targets:
// a Hilbert run of 64 points is more compact than a Morton run (no jumps
// between distant quadrants), so the 64 lanes of a traversal wave agree on
// more accept/open decisions.
TC_DEV uint32_t hilbert15(uint32_t x, uint32_t y)
{
    const uint32_t n1 = (1u << TC_LMAX) - 1u;
    uint32_t d = 0;
    for (uint32_t s = 1u << (TC_LMAX - 1); s > 0; s >>= 1) {
        const uint32_t rx = (x & s) ? 1u : 0u;
        const uint32_t ry = (y & s) ? 1u : 0u;
        d += s * s * ((3u * rx) ^ ry);
        if (ry == 0) {
            if (rx == 1) {
                x = n1 - x;
                y = n1 - y;
            }
            const uint32_t t = x;
            x = y;
            y = t;
        }
    }
    return d;
}

// ------------------------------------------------------------------ radix sort
// Stable LSD radix sort of (key, index) pairs, one launch per pass
// (k_rs_pass_lb): each tile of RS_NT IT keys is ranked stably in LDS with
// wavefront ballots, digit d of tile t is placed at (keys of smaller digits,
// from the digit totals the key kernel adds up) + (digit d in earlier tiles,
// by look-back over the counts the earlier tiles publish), and the tile's digit
// runs are written contiguously.
// Lanes of the wave holding the same digit d as this lane (among lanes
// with ok set): a lane differs from this one where, for some bit, its ballot
// bit differs from this lane's own bit.  The per-lane 0 / ~0 of each bit is a
// sign-extended bit field, so each bit costs a ballot and four 32-bit logic ops.
template <int BITS> TC_DEV unsigned long long wave_digit_peers(uint32_t d, bool ok)
{
    uint32_t diff_lo = 0, diff_hi = 0;
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
        const unsigned long long bb = tc_ballot((d >> b) & 1u);
        const uint32_t own = (uint32_t)((int32_t)(d << (31 - b)) >> 31);
        diff_lo |= (uint32_t)bb ^ own;
        diff_hi |= (uint32_t)(bb >> 32) ^ own;
    }
    const unsigned long long diff = ((unsigned long long)diff_hi << 32) | diff_lo;
    return tc_ballot(ok) & ~diff;
}

// One tile of a radix pass: the tile's keys are ranked stably in LDS and
// written out as contiguous digit runs.  start(tot, s_w) is called by every
// thread of the block after the ranking (it may use the block scratch s_w for
// collective scans); for digit threadIdx.x, of which the tile holds tot keys, it
// returns the global position of the tile's first key of that digit.  From 8 keys per
// thread on keys and indices take turns in one exchange buffer, so that two tiles
// (at 15 keys one) fit a CU's LDS.
template <int IT, class Start>
TC_DEV void rs_tile(const uint32_t *kin, const uint32_t *vin, uint32_t *kout, uint32_t *vout, int n, int shift,
                    int tile, Start &&start)
{
    constexpr int NT = RS_NT, KEYS = NT * IT, NW = NT / 64, WITEMS = 64 * IT;  // waves per tile, keys per wave
    constexpr bool TURNS = IT >= 8;
    static_assert(KEYS < 65536 && NT == RS_BINS, "16-bit counts, a thread per digit");
    __shared__ uint32_t s_k[KEYS * (TURNS ? 1 : 2)];
    uint32_t *const s_v = s_k + (TURNS ? 0 : KEYS);
    __shared__ uint32_t s_gofs[RS_BINS];                  // a digit's global start less its start in the tile
    __shared__ alignas(4) uint16_t s_wrun[NW][RS_BINS];   // per-wave digit counts, then per-wave tile offsets
    __shared__ uint32_t s_w[NW + 1];

    const int tid = threadIdx.x, lane = tc_lane(), wid = tid >> 6;
    const int base = tile * KEYS;
    const int cnt = min(KEYS, n - base);
    for (int d = lane; d < RS_BINS / 2; d += 64)
        reinterpret_cast<uint32_t *>(s_wrun[wid])[d] = 0;
    tc_wave_sync();

    // Each wave ranks its own contiguous WITEMS keys (item j of lane l is key
    // base + wid*WITEMS + 64 j + l), so the order (wave, j, lane) is the input
    // order and the ranks are stable without block barriers: peers with the
    // same digit are found with a ballot per bit, the wave's running count per
    // digit lives in s_wrun[wid] (all lanes read it before the leader updates it).
    // Bounds are tested on the offset within the tile, so base + offset is
    // only formed below n (no int overflow for n near INT_MAX).
    uint32_t k[IT], v[IT], pos[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int o = wid * WITEMS + j * 64 + lane;
        const bool ok = o < cnt;
        const int i = base + (ok ? o : 0);
        k[j] = ok ? kin[i] : 0u;
        v[j] = ok ? (vin ? vin[i] : (uint32_t)i) : 0u;
    }
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const bool ok = wid * WITEMS + j * 64 + lane < cnt;
        const uint32_t d = (k[j] >> shift) & (RS_BINS - 1);
        const unsigned long long peers = wave_digit_peers<RS_BITS>(d, ok);
        const uint32_t lower = __popcll(peers & tc_lanemask_lt());
        const uint32_t run = ok ? s_wrun[wid][d] : 0u;
        tc_wave_sync();
        if (ok && lower == 0)
            s_wrun[wid][d] = (uint16_t)(run + (uint32_t)__popcll(peers));
        tc_wave_sync();
        pos[j] = run + lower;
    }
    __syncthreads();
    {
        // digit tid: its global start, then the tile offset = exclusive scan
        // over digits of the tile counts; wave w's keys of that digit start
        // after waves 0..w-1
        uint32_t c[NW], tot = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            c[w] = s_wrun[w][tid];
            tot += c[w];
        }
        const uint32_t g = start(tot, s_w);
        uint32_t off = block_scan_excl<NT>(tot, s_w, nullptr);
        s_gofs[tid] = g - off;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            s_wrun[w][tid] = (uint16_t)off;
            off += c[w];
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        pos[j] += s_wrun[wid][(k[j] >> shift) & (RS_BINS - 1)];
        if (wid * WITEMS + j * 64 + lane < cnt) {
            s_k[pos[j]] = k[j];
            if constexpr (!TURNS)
                s_v[pos[j]] = v[j];
        }
    }
    __syncthreads();
    uint32_t dst[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int p = tid + j * NT;
        dst[j] = 0;
        if (p < cnt) {
            const uint32_t kk = s_k[p];
            dst[j] = s_gofs[(kk >> shift) & (RS_BINS - 1)] + (uint32_t)p;
            kout[dst[j]] = kk;
            if constexpr (!TURNS)
                vout[dst[j]] = s_v[p];
        }
    }
    if constexpr (TURNS) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j)
            if (wid * WITEMS + j * 64 + lane < cnt)
                s_v[pos[j]] = v[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const int p = tid + j * NT;
            if (p < cnt)
                vout[dst[j]] = s_v[p];
        }
    }
}

// Above SS_N points each pass is one launch.  The region (zeroed by
// k_bbox_partial before the keys) holds RS_PASSES x RS_BINS words, every pass's digit
// totals over all keys (k_keys_hist); one ticket per pass (64 words); and for
// each pass the tiles' published digit counts, flags[ntiles][RS_BINS]: 0 before,
// the tile's own count plus one, then LB_INC | its count plus those of all earlier
// tiles (at most the number of keys, 31 bits).
constexpr int LB_HIST = RS_PASSES * RS_BINS;
constexpr int LB_TICKETS = 64;
constexpr uint32_t LB_INC = 1u << 31;
constexpr int RS_SPIN_MAX = 1 << 22;  // polls of one unpublished count before the pass gives up
constexpr int RS_LB_BATCH = 4;        // earlier tiles' counts read per round trip

// 32-bit words of the region for a sort of ntiles tiles
static size_t lb_words(int ntiles)
{
    return (size_t)LB_HIST + LB_TICKETS + (size_t)RS_PASSES * RS_BINS * ntiles;
}

// One pass of the sort (decoupled look-back).  Tiles are taken in ticket
// order; a tile publishes its digit counts as soon as it has ranked
// its keys, then walks back over the tiles before it, adding their counts,
// until it meets one that has published LB_INC, and publishes its own LB_INC.
// A tile only ever waits for a first count, which a tile with a smaller ticket
// (started earlier) publishes without waiting: every wait ends.  Digit d of
// tile t starts at (keys of smaller digits, from hist) + (digit d in tiles
// 0..t-1), exactly as with a scan of the tile histograms.  A count that stays
// unpublished for RS_SPIN_MAX polls sets bit 1 of *err (reported by the host
// as a failed sort) and ends the walk.
template <int IT>
__global__ __launch_bounds__(RS_NT) void k_rs_pass_lb(SortSets sets, int pass)
{
    __shared__ int s_tile;
    const SortSet &t = (int)blockIdx.x < sets.s[0].ntiles ? sets.s[0] : sets.s[1];
    const uint32_t *const hist = t.lb + RS_BINS * pass;
    uint32_t *const err = t.bad;
    uint32_t *const flags = t.lb + LB_HIST + LB_TICKETS + (size_t)RS_BINS * t.ntiles * pass;
    // ping-pong scratch -> out -> scratch -> out; the first pass makes the indices
    static_assert(RS_PASSES & 1, "the keys start in the scratch");
    const bool odd = !(pass & 1);
    const uint32_t *const kin = odd ? t.k2 : t.keys, *const vin = pass == 0 ? nullptr : (odd ? t.v2 : t.perm);
    uint32_t *const kout = odd ? t.keys : t.k2, *const vout = odd ? t.perm : t.v2;
    const uint32_t before = hist[threadIdx.x];
    if (threadIdx.x == 0)
        s_tile = (int)atomicAdd(t.lb + LB_HIST + pass, 1u);
    __syncthreads();
    const int tile = s_tile;
    rs_tile<IT>(kin, vin, kout, vout, t.n, RS_BITS * pass, tile, [&](uint32_t tot, uint32_t *s_w) {
        const int d = threadIdx.x;
        uint32_t *fd = flags + d;  // fd[t * RS_BINS]: digit d of tile t
        __hip_atomic_store(&fd[(size_t)tile * RS_BINS], tile ? tot + 1u : LB_INC | tot, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        // (before the walk: the other tiles publish meanwhile)
        const uint32_t first = block_scan_excl<RS_NT>(before, s_w, nullptr);
        uint32_t pre = 0;
        bool done = tile == 0;
        int u = tile;  // tiles u .. tile-1 are summed
        while (!done) {
            // the counts of tiles u-1, u-2, ..., RS_LB_BATCH loads in flight at once
            const int nt = min(RS_LB_BATCH, u);
            uint32_t c[RS_LB_BATCH];
#pragma unroll
            for (int j = 0; j < RS_LB_BATCH; ++j)
                c[j] = j < nt ? __hip_atomic_load(&fd[(size_t)(u - 1 - j) * RS_BINS], __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : 0u;
#pragma unroll
            for (int j = 0; j < RS_LB_BATCH; ++j) {
                if (!done && j < nt) {
                    uint32_t w = c[j];
                    // tile u-1-j has not published yet: wait for it
                    for (int spin = 0; !w && spin < RS_SPIN_MAX; ++spin) {
                        __builtin_amdgcn_s_sleep(2);
                        w = __hip_atomic_load(&fd[(size_t)(u - 1 - j) * RS_BINS], __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
                    }
                    if (!w)
                        atomicOr(err, 2u);
                    pre += w & LB_INC ? w & ~LB_INC : w ? w - 1u : 0u;
                    done = (w & LB_INC) || !w;
                }
            }
            u -= nt;
        }
        if (tile)
            __hip_atomic_store(&fd[(size_t)tile * RS_BINS], LB_INC | (pre + tot), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        return first + pre;
    });
}

// Keys of the points: sources by sort-sources.cpp:87-110 (quantise +
// interleave, x in even bits), with `packed` also the source record
// {x, y, v, 0} in input order, so the gather after the sort reads one 32-byte
// record per source; targets by hilbert15.  Steps of kstep points (a multiple of
// 1,024) are taken in turn by a set's kgrid workgroups, and each workgroup adds the
// digit totals of all passes into lb (zeroed before) once.  Each
// workgroup finishes the bounding box from k_bbox_partial's np partials and
// per-workgroup flags itself (a set's first one writes it and the non-finite flag).
__global__ __launch_bounds__(256) void k_keys_hist(SortSets sets)
{
    __shared__ uint32_t h[LB_HIST];
    __shared__ double s_box[4];
    const bool second = (int)blockIdx.x >= sets.s[0].kgrid;
    const SortSet &t = second ? sets.s[1] : sets.s[0];
    const int bi = blockIdx.x - (second ? sets.s[0].kgrid : 0), n = t.n, step = t.kstep;
    const double *x = t.x, *y = t.y, *v = t.v;
    for (int i = threadIdx.x; i < LB_HIST; i += 256)
        h[i] = 0;
    if (threadIdx.x < 64)
        bbox_finish(t.part, t.np, s_box);
    __syncthreads();
    if (bi == 0 && threadIdx.x < 64) {
        uint32_t b = 0;
        for (int i = threadIdx.x; i < t.np; i += 64)
            b |= t.pbad[i];
        b = tc_ballot(b != 0) ? 1u : 0u;
        if (threadIdx.x == 0) {
            for (int q = 0; q < 4; ++q)
                t.box[q] = s_box[q];
            *t.bad = b;
        }
    }
    const double xmin = s_box[0], ymin = s_box[1], scale = s_box[3];
    // four points a turn, loaded before the first is stored (the compiler cannot
    // tell the arrays apart)
    constexpr int U = 4;
    static_assert(KH_TILE_MIN % (256 * U) == 0 && KH_TILE_MAX % (256 * U) == 0, "whole turns");
    for (long long base = (long long)bi * step; base < n; base += (long long)t.kgrid * step) {
        for (int j = 0; j < step; j += 256 * U) {
            const long long i0 = base + j + threadIdx.x;
            double xi[U], yi[U], vi[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const long long i = i0 + 256 * u;
                xi[u] = i < n ? x[i] : 0.0;
                yi[u] = i < n ? y[i] : 0.0;
                vi[u] = i < n && t.packed ? v[i] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const long long i = i0 + 256 * u;
                if (i >= n)
                    break;
                const uint32_t qx = quantise(xi[u], xmin, scale), qy = quantise(yi[u], ymin, scale);
                const uint32_t k = v ? tc_spread15(qx) | (tc_spread15(qy) << 1) : hilbert15(qx, qy);
                t.k2[i] = k;
                if (t.packed)
                    t.packed[i] = make_double4(xi[u], yi[u], vi[u], 0.0);
#pragma unroll
                for (int q = 0; q < RS_PASSES; ++q)
                    atomicAdd(&h[q * RS_BINS + ((k >> (RS_BITS * q)) & (RS_BINS - 1))], 1u);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < LB_HIST; i += 256)
        if (h[i])
            atomicAdd(&t.lb[i], h[i]);
}

// ------------------------------------------------------------------ small sorts
// Up to SS_N points in one workgroup: bounding box (k_bbox_partial +
// bbox_finish semantics), keys (Morton or Hilbert as k_keys_hist), the same
// stable 4-pass LSD radix sort as above with the keys in registers and each
// pass's scatter in LDS, and for sources the gather of the sorted records.
// One launch instead of seven (and for two sets instead of fourteen), which is what
// a small solve is made of.  IT keys
// per thread, the least of 1, 2, 4, 8, 12, 16 that holds the points: the ranking (8
// ballots per key slot and pass) is what the kernel spends its time on, and
// with 16 slots for every n it took 48 us at 1,000 points and 79 us at 10,000,
// with the points on one wave instead of 16; 15 us now at 1,000 points, and back
// to back on warm caches 43 -> 13.5 us at 1,000, 44 -> 22 at 4,000, 47 -> 33 at 8,000.
constexpr int SS_NT = 1024, SS_MAX_IT = 16, SS_N = SS_NT * SS_MAX_IT;
static_assert(SS_N == TC_SORT_SMALL_MAX, "one-workgroup sort size");

// The one-workgroup sort of one point set (the body of k_sort_small and of
// k_sort_small_batch's workgroups); the sorted keys stay in lds.k.
template <int IT> struct SortSmallLds {
    uint32_t k[SS_NT * IT], v[SS_NT * IT], wrun[SS_NT / 64][SS_BINS];
};
template <int IT>
TC_DEV void sort_small(SortSmallLds<IT> &lds, bool hilbert, const double *__restrict__ x,
                       const double *__restrict__ y, const double *__restrict__ v, int n,
                       double *__restrict__ box_out, uint32_t *__restrict__ bad_out,
                       uint32_t *__restrict__ keys_out, uint32_t *__restrict__ perm_out,
                       double4 *__restrict__ src_out)
{
    constexpr int NW = SS_NT / 64, WITEMS = 64 * IT;
    uint32_t *const s_k = lds.k, *const s_v = lds.v;
    uint32_t(*const s_wrun)[SS_BINS] = lds.wrun;
    __shared__ uint32_t s_w[NW + 1];
    __shared__ double4 s_red[NW];
    __shared__ double s_box[4];
    __shared__ uint32_t s_bad[NW];
    const int tid = threadIdx.x, lane = tc_lane(), wid = tid >> 6;

    // this thread's points, item j of lane l of wave w being position
    // w * WITEMS + 64 j + l (all loads in flight at once)
    double xr[IT], yr[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int i = wid * WITEMS + j * 64 + lane;
        xr[j] = i < n ? x[i] : 0.0;
        yr[j] = i < n ? y[i] : 0.0;
    }
    // bounding box: max accumulators start at 0 as in the reference
    double xmi = 1e13, ymi = 1e13, xma = 0, yma = 0;
    bool nonfinite = false;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int i = wid * WITEMS + j * 64 + lane;
        if (i < n) {
            const double a = xr[j], b = yr[j];
            nonfinite |= !isfinite(a) || !isfinite(b);
            xmi = a < xmi ? a : xmi;
            xma = xma < a ? a : xma;
            ymi = b < ymi ? b : ymi;
            yma = yma < b ? b : yma;
        }
    }
    tc_wave_box(xmi, ymi, xma, yma);
    const bool wbad = tc_ballot(nonfinite) != 0;
    if (lane == 0) {
        s_red[wid] = make_double4(xmi, xma, ymi, yma);
        s_bad[wid] = wbad ? 1u : 0u;
    }
    __syncthreads();
    if (tid == 0) {
        double4 r = s_red[0];
        uint32_t bad = s_bad[0];
        for (int w = 1; w < NW; ++w) {
            r.x = s_red[w].x < r.x ? s_red[w].x : r.x;
            r.y = r.y < s_red[w].y ? s_red[w].y : r.y;
            r.z = s_red[w].z < r.z ? s_red[w].z : r.z;
            r.w = r.w < s_red[w].w ? s_red[w].w : r.w;
            bad |= s_bad[w];
        }
        const double ext0 = r.y - r.x, ext1 = r.w - r.z;
        const double eps = 10000 * DBL_EPSILON;
        double ext = (ext0 < ext1 ? ext1 : ext0) * (1 + 2 * eps);
        if (!(ext > 0))
            ext = 1.0;
        s_box[0] = r.x - eps * ext;
        s_box[1] = r.z - eps * ext;
        s_box[2] = ext;
        s_box[3] = (1.0 / ext) * (double)(1 << TC_LMAX);
        for (int q = 0; q < 4; ++q)
            box_out[q] = s_box[q];
        *bad_out = bad;
    }
    __syncthreads();

    const double xmin = s_box[0], ymin = s_box[1], scale = s_box[3];
    uint32_t k[IT], vi[IT], dr[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int i = wid * WITEMS + j * 64 + lane;
        const uint32_t qx = quantise(xr[j], xmin, scale), qy = quantise(yr[j], ymin, scale);
        k[j] = i < n ? (hilbert ? hilbert15(qx, qy) : (tc_spread15(qx) | (tc_spread15(qy) << 1))) : 0u;
        vi[j] = (uint32_t)i;
    }

#pragma unroll 1
    for (int shift = 0;; shift += 8) {
        for (int d = lane; d < SS_BINS; d += 64)
            s_wrun[wid][d] = 0;
        tc_wave_sync();
        // wave-local stable ranks, as in rs_tile
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const bool ok = wid * WITEMS + j * 64 + lane < n;
            const uint32_t d = (k[j] >> shift) & (SS_BINS - 1);
            const unsigned long long peers = wave_digit_peers<8>(d, ok);
            const uint32_t lower = __popcll(peers & tc_lanemask_lt());
            const uint32_t run = ok ? s_wrun[wid][d] : 0u;
            tc_wave_sync();
            if (ok && lower == 0)
                s_wrun[wid][d] = run + (uint32_t)__popcll(peers);
            tc_wave_sync();
            dr[j] = ((run + lower) << 8) | d;
        }
        __syncthreads();
        {
            // digit tid: start = exclusive scan of the digit totals; wave w's
            // keys of that digit follow waves 0..w-1
            uint32_t c[NW], tot = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                c[w] = tid < SS_BINS ? s_wrun[w][tid] : 0u;
                tot += c[w];
            }
            uint32_t off = block_scan_excl<SS_NT>(tot, s_w, nullptr);
            if (tid < SS_BINS) {
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    s_wrun[w][tid] = off;
                    off += c[w];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            if (wid * WITEMS + j * 64 + lane < n) {
                const uint32_t pos = s_wrun[wid][dr[j] & 255u] + (dr[j] >> 8);
                s_k[pos] = k[j];
                s_v[pos] = vi[j];
            }
        }
        __syncthreads();
        if (shift == 24)
            break;
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            const int p = wid * WITEMS + j * 64 + lane;
            if (p < n) {
                k[j] = s_k[p];
                vi[j] = s_v[p];
            }
        }
    }

#pragma unroll 8
    for (int p = tid; p < n; p += SS_NT) {
        const uint32_t i = s_v[p];
        keys_out[p] = s_k[p];
        perm_out[p] = i;
        if (src_out)
            src_out[p] = make_double4(x[i], y[i], v[i], 0.0);
    }
}

// Target orders of several requests at once: workgroup b sorts desc[b]'s
// targets as k_sort_small does alone (the order does not depend on IT).
template <int IT> __global__ __launch_bounds__(SS_NT) void k_sort_small_batch(const TcSortDesc *__restrict__ desc)
{
    __shared__ SortSmallLds<IT> lds;
    const TcSortDesc &d = desc[blockIdx.x];
    sort_small<IT>(lds, true, d.x, d.y, nullptr, d.n, d.box, d.bad, d.keys, d.perm, nullptr);
}

// f(std::integral_constant<int, IT>) with the least IT whose SS_NT IT slots hold n points.
template <class F> void small_items(int n, F &&f)
{
    if (n <= SS_NT)
        f(std::integral_constant<int, 1>());
    else if (n <= 2 * SS_NT)
        f(std::integral_constant<int, 2>());
    else if (n <= 4 * SS_NT)
        f(std::integral_constant<int, 4>());
    else if (n <= 8 * SS_NT)
        f(std::integral_constant<int, 8>());
    else if (n <= 12 * SS_NT)
        f(std::integral_constant<int, 12>());
    else
        f(std::integral_constant<int, SS_MAX_IT>());
}

__global__ __launch_bounds__(256) void k_gather_src(const double4 *packed, const uint32_t *perm, int n,
                                                     double4 *src)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n)
        return;
    src[i] = packed[perm[i]];
}

// ------------------------------------------------------------------ topology
// Internal cells are exactly the cells of levels 0..14 holding more than
// `cap` sources (their ancestors then hold more too), i.e. the breadth-first
// build_tree recursion of upward.cpp:223-277.  A level-L cell starting at
// sorted position i is internal iff key[i-1] leaves the cell and key[i+cap]
// stays in it, so every internal cell is found from three key reads, and its
// breadth-first rank is a scan over (level, position).
// A wave covers 64 IT consecutive positions, item j of lane l being position
// base + 64 j + l; all the keys it needs are requested before the first is
// used (one memory round trip per wave instead of IT).  Few items per wave where
// the positions are few (more waves, shorter chains), many where they fill the
// GPU anyway and the census table (TC_LMAX counts per workgroup) should stay
// short.  Count and emission at 65,536 positions, key by key with IT = 16: 11 +
// 16 us, with IT = 4: 5 + 6 us; at 2^24 positions 49 + 73 us, with IT = 16: 30 + 60 us.
constexpr int TB_IT_SMALL = 4, TB_IT = 16, TB_SMALL_N = 1 << 20;

// Census record: level starts, internal count, non-finite flags of the sources and of
// targets sorted with them (info in device memory), and at int offset INFO_BOX the
// bounding box; the kernels write it to pinned host memory too, so no copy is queued.
constexpr int INFO_BOX = 20;
constexpr size_t INFO_BYTES = sizeof(int) * INFO_BOX + sizeof(double) * 4;

// Internal levels [lo, hi] of the cells starting at this lane's positions
// (none where hi < lo).
template <int IT> TC_DEV void cell_ranges(const uint32_t *keys, int n, int cap, int base, int (&lo)[IT], int (&hi)[IT])
{
    uint32_t k[IT], kp[IT], kc[IT];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int i = base + 64 * j + tc_lane();
        k[j] = i < n ? keys[i] : 0u;
        kp[j] = i < n && i > 0 ? keys[i - 1] : 0u;
        kc[j] = i + cap < n ? keys[i + cap] : 0u;
    }
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int i = base + 64 * j + tc_lane();
        lo[j] = i >= n ? 1 : (i == 0 ? 0 : tc_common_level(kp[j], k[j]) + 1);
        hi[j] = i >= n ? 0 : (i + cap < n ? min(TC_LMAX - 1, tc_common_level(k[j], kc[j])) : -1);
    }
}

// The workgroup's internal cells per level: into s_cnt[wave][level].
template <int IT> TC_DEV void cell_counts(const int (&lo)[IT], const int (&hi)[IT], uint32_t (*s_cnt)[TC_LMAX])
{
    uint32_t c[TC_LMAX];
#pragma unroll
    for (int L = 0; L < TC_LMAX; ++L)
        c[L] = 0;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        if (!tc_ballot(hi[j] >= lo[j]))
            continue;
#pragma unroll
        for (int L = 0; L < TC_LMAX; ++L)
            c[L] += __popcll(tc_ballot(L >= lo[j] && L <= hi[j]));
    }
    if (tc_lane() == 0)
#pragma unroll
        for (int L = 0; L < TC_LMAX; ++L)
            s_cnt[threadIdx.x >> 6][L] = c[L];
    __syncthreads();
}

template <int IT>
__global__ __launch_bounds__(256) void k_int_count(const uint32_t *keys, int n, int cap, uint32_t *cnt_tab,
                                                    int stride)
{
    __shared__ uint32_t s_cnt[4][TC_LMAX];
    const int base = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 64 * IT;
    int lo[IT], hi[IT];
    cell_ranges<IT>(keys, n, cap, base, lo, hi);
    cell_counts<IT>(lo, hi, s_cnt);
    if (threadIdx.x < TC_LMAX)
        cnt_tab[(size_t)threadIdx.x * stride + blockIdx.x] =
            s_cnt[0][threadIdx.x] + s_cnt[1][threadIdx.x] + s_cnt[2][threadIdx.x] + s_cnt[3][threadIdx.x];
}

// The census in one workgroup: cnt holds TC_LMAX rows (levels) of nblk counts,
// `stride` (a multiple of 4) apart; wave L sums, then scans row L, 1,024 counts
// a step, so the rows run side by side, each step is one round of wide loads
// and no count needs its level by division.  Writes every block's first rank
// per level (level-major breadth-first order) to offs and the census record.
// 4,096 blocks (2^24 positions): 11 us; the scan over all rows as one array
// took 25 us in four launches.
__global__ __launch_bounds__(SCAN_NT) void k_census(const uint32_t *cnt, uint32_t *offs, int nblk, int stride,
                                                     const uint32_t *bad, const uint32_t *tbad, const double *box,
                                                     int *info, int *hinfo)
{
    static_assert(TC_LMAX < SCAN_NT / 64, "one wave per level");
    __shared__ uint32_t s_tot[SCAN_NT / 64];
    const int lane = tc_lane(), L = threadIdx.x >> 6;
    // 16 counts of this lane from step b0: positions b0 + 256 j + 4 lane .. + 3
    auto load = [&](int b0, uint4 (&v)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int b = b0 + 256 * j + 4 * lane;
            v[j] = b < nblk ? *reinterpret_cast<const uint4 *>(cnt + (size_t)L * stride + b) : make_uint4(0, 0, 0, 0);
            v[j].y = b + 1 < nblk ? v[j].y : 0u;  // a row's last words may be padding
            v[j].z = b + 2 < nblk ? v[j].z : 0u;
            v[j].w = b + 3 < nblk ? v[j].w : 0u;
        }
    };
    uint32_t tot = 0;
    if (L < TC_LMAX)
        for (int b0 = 0; b0 < nblk; b0 += 1024) {
            uint4 v[4];
            load(b0, v);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                tot += (v[j].x + v[j].y) + (v[j].z + v[j].w);
        }
    tc_offsets<32, 1>([&](auto off) { tot = tc_xor_add<off.value>(tot); });
    if (lane == 0)
        s_tot[L] = tot;
    __syncthreads();
    uint32_t start = 0;
    for (int q = 0; q < L; ++q)
        start += s_tot[q];
    if (lane == 0) {
        auto put = [&](int at, int v) {
            info[at] = v;
            __hip_atomic_store(hinfo + at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        };
        if (L <= TC_LMAX)
            put(L, (int)start);  // row TC_LMAX: the total
        if (L == 0) {
            put(TC_LMAX + 1, (int)*bad);
            put(TC_LMAX + 2, tbad ? (int)*tbad : 0);
        }
    }
    if (threadIdx.x >= 32 && threadIdx.x < 36)
        __hip_atomic_store(reinterpret_cast<double *>(hinfo + INFO_BOX) + (threadIdx.x - 32), box[threadIdx.x - 32],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (L >= TC_LMAX)
        return;
    for (int b0 = 0; b0 < nblk; b0 += 1024) {
        uint4 v[4];
        load(b0, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t sum = (v[j].x + v[j].y) + (v[j].z + v[j].w);
            const uint32_t x = tc_wave_scan(sum);
            const int b = b0 + 256 * j + 4 * lane;
            uint4 o;
            o.x = start + x - sum;
            o.y = o.x + v[j].x;
            o.z = o.y + v[j].y;
            o.w = o.z + v[j].z;
            if (b < nblk)  // within the padded row
                *reinterpret_cast<uint4 *>(offs + (size_t)L * stride + b) = o;
            start += (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
        }
    }
}

template <int IT>
__global__ __launch_bounds__(256) void k_int_emit(const uint32_t *keys, int n, int cap, const uint32_t *offs,
                                                   int stride, int tmax, int *istart, int *ilevel)
{
    __shared__ uint32_t s_cnt[4][TC_LMAX];
    const int wid = threadIdx.x >> 6;
    const int base = (blockIdx.x * 4 + wid) * 64 * IT;
    uint32_t c[TC_LMAX];
#pragma unroll
    for (int L = 0; L < TC_LMAX; ++L)
        c[L] = offs[(size_t)L * stride + blockIdx.x];
    int lo[IT], hi[IT];
    cell_ranges<IT>(keys, n, cap, base, lo, hi);
    cell_counts<IT>(lo, hi, s_cnt);
#pragma unroll
    for (int L = 0; L < TC_LMAX; ++L)
        for (int w = 0; w < wid; ++w)
            c[L] += s_cnt[w][L];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        if (!tc_ballot(hi[j] >= lo[j]))
            continue;
#pragma unroll
        for (int L = 0; L < TC_LMAX; ++L) {
            const bool f = L >= lo[j] && L <= hi[j];
            const unsigned long long b = tc_ballot(f);
            if (f) {
                const uint32_t r = c[L] + __popcll(b & tc_lanemask_lt());
                if (r < (uint32_t)tmax) {
                    istart[r] = base + 64 * j + tc_lane();
                    ilevel[r] = L;
                }
            }
            c[L] += __popcll(b);
        }
    }
}

constexpr int NODES_WAVE_T = 16384;
// Internal nodes of the tree being built, from its census record; the buffers hold
// tmax.  None where the sort failed (bit 1 of the flag): the keys are then in no order.
TC_DEV int census_nodes(const int *__restrict__ info, int tmax)
{
    return info[TC_LMAX + 1] & 2 ? 0 : min(info[TC_LMAX], tmax);
}

// First position in [lo, hi) where pred is false (pred holds on a prefix of
// the range), searched by a group of G lanes that hold the same range: G evenly
// spread probes a round, one memory access each.
template <int G> TC_DEV int group_count(bool ok)
{
    return __popcll((tc_ballot(ok) >> (tc_lane() & ~(G - 1))) & (G == 64 ? ~0ull : (1ull << G) - 1ull));
}
template <int G, class Pred> TC_DEV int group_partition(int lo, int hi, Pred &&pred)
{
    while (hi > lo) {
        const int step = (hi - lo + G - 1) / G;
        const int p = lo + (tc_lane() & (G - 1)) * step;
        const int c = group_count<G>(p < hi && pred(p));
        if (c == 0)
            return lo;
        const int last = lo + (c - 1) * step;  // the last probe where it held
        hi = min(hi, last + step);
        lo = last + 1;
    }
    return lo;
}

// One internal node (breadth-first rank r) per group of G lanes: its id from
// its parent's rank, the end of its cell, the ranges of its four children.  A
// search by one thread is a chain of some 70 dependent loads (22 us at 2^16, 56
// us at 2^24 sources whatever the leaf size).  By a wave (G = 64) it is about
// 8 rounds, the shortest chain, taken while the nodes are too few to fill the
// GPU; beyond NODES_WAVE_T nodes, 16 lanes a node keep four times as many searches in
// flight.  2^16 sources: 22 -> 7 us, 2^20: 31 -> 13 us (G = 64), 2^23: 38 -> 33 us
// (G = 16).  Every node writes its children's records; a child that
// is internal writes its own child field (its rank is its own), so only leaves'
// are cleared here.  Leaves the parent's rank in ilevel and the count of
// internal children in pend for the upward pass.
template <int G>
__global__ __launch_bounds__(256) void k_int_nodes(const uint32_t *__restrict__ keys, int n, int cap,
                                                    const int *__restrict__ istart, int *ilevel,
                                                    const int *__restrict__ info, int tmax, int *__restrict__ selfid,
                                                    uint32_t *pend, uint32_t *child, int2 *se, int *level, int2 *cell)
{
    const int r = blockIdx.x * (256 / G) + threadIdx.x / G, lane = threadIdx.x % G;
    const int T = census_nodes(info, tmax);
    if (T == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
        // a tree of one leaf
        child[0] = 0u;
        se[0] = make_int2(0, n);
        level[0] = 0;
        cell[0] = make_int2(0, 0);
    }
    if (r >= T)
        return;
    const int L = ilevel[r], i = istart[r];
    const uint32_t key = keys[i];
    const int sh = 2 * (TC_LMAX - L);
    const uint32_t prefix = key >> sh;  // sh <= 30
    int self = 0, up = 0, e = n;
    if (L > 0) {
        // the parent: the last internal cell of level L - 1 starting at or before i
        const int l0 = info[L - 1];
        up = group_partition<G>(l0, info[L], [&](int p) { return istart[p] <= i; }) - 1;
        self = 1 + 4 * up + (int)(prefix & 3u);
        // the cell's end: bracketed by doubling steps, one lane each
        const int b0 = i + cap + 1;  // the cell holds more than cap sources
        constexpr int NP = G < 30 ? G : 30;
        const int o = lane < NP ? (1 << lane) - 1 : INT_MAX;
        const bool in = o < n - b0 && (keys[b0 + o] >> sh) == prefix;
        const int c = group_count<G>(in);  // probes 0 .. c-1 lie inside
        const int lo = c ? b0 + (1 << (c - 1)) : b0;
        const int hi = c < NP ? (int)min((long long)n, (long long)b0 + (1ll << c) - 1) : n;
        e = group_partition<G>(lo, hi, [&](int p) { return (keys[p] >> sh) == prefix; });
    }
    if (lane == 0) {
        selfid[r] = self;
        ilevel[r] = up;  // read by this wave alone, above
        child[self] = (uint32_t)(1 + 4 * r);
        if (L == 0) {
            se[0] = make_int2(0, n);
            level[0] = 0;
            cell[0] = make_int2(0, 0);
        }
    }
    const int csh = sh - 2;
    int b[5];
    b[0] = i;
    b[4] = e;
#pragma unroll
    for (int c = 1; c < 4; ++c) {
        const uint32_t target = ((prefix << 2) | (uint32_t)c) << csh;
        b[c] = group_partition<G>(b[c - 1], e, [&](int p) { return keys[p] < target; });
    }
    bool inner = false;
    if (lane < 4) {
        const int cs = lane == 0 ? b[0] : (lane == 1 ? b[1] : (lane == 2 ? b[2] : b[3]));
        const int ce = lane == 0 ? b[1] : (lane == 1 ? b[2] : (lane == 2 ? b[3] : b[4]));
        const int k = 1 + 4 * r + lane;
        se[k] = make_int2(cs, ce);
        level[k] = L + 1;
        cell[k] = make_int2(2 * (int)tc_compact15(prefix) + (lane & 1), 2 * (int)tc_compact15(prefix >> 1) + (lane >> 1));
        inner = ce - cs > cap && L + 1 < TC_LMAX;
        if (!inner)
            child[k] = 0u;
    }
    const uint32_t ni = (uint32_t)group_count<G>(inner);
    if (lane == 0)
        pend[r] = ni << 8 | ni;
}

// The whole topology of a small tree by the workgroup that sorted its keys, from
// the keys in LDS (count, census, emission and nodes of the kernels above, which
// take larger trees): a launch each costs the host more than this takes.
// At most tmax <= SMALL_TOPO_T internal nodes, a thread per node: a search is a
// chain of LDS reads, about 50 ns each.  With the joint
// sorts, 1,000 points drop-in: 138 -> 105 us; 31,623 on host arrays 388 -> 329 us.
constexpr int SMALL_TOPO_T = SS_NT;
struct SmallTopo {
    int cap, tmax;  // tmax 0: no topology
    int *info, *hinfo, *selfid, *parent;
    uint32_t *pend, *child;
    int2 *se;
    int *level;
    int2 *cell;
};

template <int IT>
TC_DEV void small_topology(SortSmallLds<IT> &lds, const SmallTopo &tp, int n, const double *box, const uint32_t *bad)
{
    constexpr int NW = SS_NT / 64;
    static_assert(SS_N <= 1 << 14 && TC_LMAX < 16, "position and level share a word");
    const int tid = threadIdx.x, lane = tc_lane(), wid = tid >> 6, cap = tp.cap;
    const uint32_t *const key = lds.k;
    uint32_t *const ist = lds.v;             // position | level << 14 by breadth-first rank
    uint32_t(*const cnt)[SS_BINS] = lds.wrun;  // [wave][level], then first ranks
    __shared__ int s_start[TC_LMAX + 1];
    __syncthreads();  // the sort's last reads of lds.v and lds.wrun
    int lo[IT], hi[IT];
    uint32_t c[TC_LMAX];
#pragma unroll
    for (int L = 0; L < TC_LMAX; ++L)
        c[L] = 0;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        const int i = wid * 64 * IT + 64 * j + lane;
        const uint32_t k = i < n ? key[i] : 0u;
        lo[j] = i >= n ? 1 : (i == 0 ? 0 : tc_common_level(key[i - 1], k) + 1);
        hi[j] = i >= n ? 0 : (i + cap < n ? min(TC_LMAX - 1, tc_common_level(k, key[i + cap])) : -1);
        if (!tc_ballot(hi[j] >= lo[j]))
            continue;
#pragma unroll
        for (int L = 0; L < TC_LMAX; ++L)
            c[L] += __popcll(tc_ballot(L >= lo[j] && L <= hi[j]));
    }
    if (lane == 0)
#pragma unroll
        for (int L = 0; L < TC_LMAX; ++L)
            cnt[wid][L] = c[L];
    __syncthreads();
    if (wid == 0) {
        // lane L: level L's count, its first rank, and each wave's
        uint32_t w[NW], tot = 0;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            w[q] = lane < TC_LMAX ? cnt[q][lane] : 0u;
            tot += w[q];
        }
        uint32_t start = tc_wave_scan(tot) - tot;
        if (lane <= TC_LMAX) {
            s_start[lane] = min((int)start, tp.tmax);
            tp.info[lane] = (int)start;
            __hip_atomic_store(tp.hinfo + lane, (int)start, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (lane < TC_LMAX)
#pragma unroll
            for (int q = 0; q < NW; ++q) {
                cnt[q][lane] = start;
                start += w[q];
            }
        if (lane == 0) {
            tp.info[TC_LMAX + 1] = (int)*bad;
            __hip_atomic_store(tp.hinfo + TC_LMAX + 1, (int)*bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        if (lane >= 32 && lane < 36)
            __hip_atomic_store(reinterpret_cast<double *>(tp.hinfo + INFO_BOX) + (lane - 32), box[lane - 32],
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __syncthreads();
#pragma unroll
    for (int L = 0; L < TC_LMAX; ++L)
        c[L] = cnt[wid][L];
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        if (!tc_ballot(hi[j] >= lo[j]))
            continue;
#pragma unroll
        for (int L = 0; L < TC_LMAX; ++L) {
            const bool f = L >= lo[j] && L <= hi[j];
            const unsigned long long b = tc_ballot(f);
            const uint32_t r = c[L] + __popcll(b & tc_lanemask_lt());
            if (f && r < (uint32_t)tp.tmax)
                ist[r] = (uint32_t)(wid * 64 * IT + 64 * j + lane) | (uint32_t)L << 14;
            c[L] += __popcll(b);
        }
    }
    __syncthreads();
    if (tid == 0) {
        // the root; without internal nodes a leaf
        tp.se[0] = make_int2(0, n);
        tp.level[0] = 0;
        tp.cell[0] = make_int2(0, 0);
        if (s_start[TC_LMAX] == 0)
            tp.child[0] = 0u;
    }
    const int r = tid;
    if (r >= s_start[TC_LMAX])
        return;
    // first position in [a, b) where pred is false
    auto partition = [](int a, int b, auto pred) {
        while (a < b) {
            const int mid = (a + b) >> 1;
            if (pred(mid))
                a = mid + 1;
            else
                b = mid;
        }
        return a;
    };
    const int L = (int)(ist[r] >> 14), i = (int)(ist[r] & 0x3fffu);
    const int sh = 2 * (TC_LMAX - L), csh = sh - 2;
    const uint32_t prefix = key[i] >> sh;
    int self = 0, up = 0, e = n;
    if (L > 0) {
        up = partition(s_start[L - 1], s_start[L], [&](int p) { return (int)(ist[p] & 0x3fffu) <= i; }) - 1;
        self = 1 + 4 * up + (int)(prefix & 3u);
        e = partition(i + cap + 1, n, [&](int p) { return (key[p] >> sh) == prefix; });
    }
    tp.selfid[r] = self;
    tp.parent[r] = up;
    tp.child[self] = (uint32_t)(1 + 4 * r);
    uint32_t inner = 0;
    int a = i;
    const int cx = 2 * (int)tc_compact15(prefix), cy = 2 * (int)tc_compact15(prefix >> 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t next = ((prefix << 2) | (uint32_t)(q + 1)) << csh;
        const int b = q == 3 ? e : partition(a, e, [&](int p) { return key[p] < next; });
        const int k = 1 + 4 * r + q;
        tp.se[k] = make_int2(a, b);
        tp.level[k] = L + 1;
        tp.cell[k] = make_int2(cx + (q & 1), cy + (q >> 1));
        if (b - a > cap && L + 1 < TC_LMAX)
            ++inner;
        else
            tp.child[k] = 0u;
        a = b;
    }
    tp.pend[r] = inner << 8 | inner;
}

// One workgroup per set (one or two): the sort and, for the first set's keys, the topology.
template <int IT>
__global__ __launch_bounds__(SS_NT) void k_sort_small(SortSets sets, double4 *__restrict__ src_out, SmallTopo tp)
{
    __shared__ SortSmallLds<IT> lds;
    const SortSet &t = blockIdx.x ? sets.s[1] : sets.s[0];
    sort_small<IT>(lds, t.v == nullptr, t.x, t.y, t.v, t.n, t.box, t.bad, t.keys, t.perm, blockIdx.x ? nullptr : src_out);
    if (tp.tmax) {
        __syncthreads();  // the box and flag written by thread 0 of this workgroup
        if (blockIdx.x == 0)
            small_topology<IT>(lds, tp, t.n, t.box, t.bad);
        else if (threadIdx.x == 0)
            __hip_atomic_store(tp.hinfo + TC_LMAX + 2, (int)*t.bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ------------------------------------------------------------------ upward
// One wavefront per leaf: build_leaf (upward.cpp:61-93) = upward_setup
// (upward-common.ispc:13-57) + upward_p2e (upward-kernels.m4:52-92), in the
// canonical 64-lane strided order with the pairwise lane tree.  What bounds it is
// the chain of a wave's memory round trips (entries, sources, and the sources
// again for the radius and for the coefficients) against the waves in flight: with the
// entries in one round and the first source of a lane kept, order 9 at 2^24 points went
// 352 -> 285 us, order 8 at 2^23 points (leaves of 64) 153 -> 129 us.  High orders would take a wave
// of occupancy more for it than they had (order 24: 160 registers, 15.0 us at 200,000
// points) and are held to it, at the price of a few spills (14.2; 13.8 before).
template <int P>
__global__ __launch_bounds__(256, P <= 16 ? 1 : P <= 24 ? 4 : 3) void k_leaf_upward(const uint32_t *child, const int2 *se, const int *level,
                                                      const int2 *cell, const double4 *src, const double *box,
                                                      const int *__restrict__ info, int tmax, TcNode *nodes, double *exps, double *dexps,
                                                      double4 *nodew, float4 *src32)
{
    const int id = tc_uniform((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    // the node's entries in one round of scalar loads (those past the tree's nodes
    // are read inside the arrays, and dropped)
    const int at = min(id, 4 * tmax);
    const uint32_t inner = child[at];
    const int2 r = se[at];
    const int l = level[at];
    const int2 cc = cell[at];
    if (id > 4 * census_nodes(info, tmax) || inner != 0)
        return;
    const int lane = tc_lane();
    const int s = r.x, e = r.y;
    const double xmin = box[0], ymin = box[1], ext = box[2];
    const double h = ext / (double)(1 << l);
    const double x0 = xmin + h * (double)cc.x, y0 = ymin + h * (double)cc.y;

    // the lane's first source stays in registers for the three sums (most leaves
    // have no second one); without one, zeros that change no sum
    const bool has = s + lane < e;
    const double4 q0 = has ? src[s + lane] : make_double4(0, 0, 0, 0);
    const double a0 = fabs(q0.z);
    double pm = q0.z, pw = a0, px = q0.x * a0, py = q0.y * a0;
    for (int i = s + lane + 64; i < e; i += 64) {
        const double4 q = src[i];
        const double a = fabs(q.z);
        pm += q.z;
        pw += a;
        px += q.x * a;
        py += q.y * a;
    }
    // lane 0: mass, 16: w, 32: wx, 48: wy (bit-identical to four tree sums)
    double g4[4] = {pm, pw, px, py};
    int first, end;
    const double gsum = tc_wave_scatter_sum<4>(g4, first, end);
    const double m = tc_lane_value(gsum, 0), w = tc_lane_value(gsum, 16);
    const double wx = tc_lane_value(gsum, 32), wy = tc_lane_value(gsum, 48);
    const double xc = w != 0 ? wx / w : (x0 + 0.5 * h);
    const double yc = w != 0 ? wy / w : (y0 + 0.5 * h);

    const double xr0 = has ? q0.x - xc : 0.0, yr0 = has ? q0.y - yc : 0.0;
    double r2 = xr0 * xr0 + yr0 * yr0;
    r2 = 0 < r2 ? r2 : 0;
    for (int i = s + lane + 64; i < e; i += 64) {
        const double4 q = src[i];
        const double xr = q.x - xc, yr = q.y - yc;
        const double d = xr * xr + yr * yr;
        r2 = r2 < d ? d : r2;
    }
    r2 = tc_wave_max(r2);
    const double rad = sqrt(r2);

    double re[P], im[P];
#pragma unroll
    for (int k = 0; k < P; ++k)
        re[k] = im[k] = 0;
    const auto add = [&](int i, double r0, double i0, double v) {
        double rtmp = r0 * v, itmp = i0 * v;
        re[0] -= rtmp;
        im[0] -= itmp;
        double rprod = r0, iprod = i0;
#pragma unroll
        for (int k = 1; k < P; ++k) {
            rtmp = rprod * r0 - iprod * i0;
            itmp = rprod * i0 + iprod * r0;
            const double term = v * (1.0 / (double)(k + 1));
            rprod = rtmp;
            iprod = itmp;
            rtmp = rprod * term;
            itmp = iprod * term;
            re[k] -= rtmp;
            im[k] -= itmp;
        }
        if (src32 && i < e)
            src32[i] = make_float4((float)r0, (float)i0, (float)v, 0.f);
    };
    add(s + lane, xr0, yr0, q0.z);
    for (int i = s + lane + 64; i < e; i += 64) {
        const double4 q = src[i];
        add(i, q.x - xc, q.y - yc, q.z);
    }
    double *ex = exps + (size_t)2 * P * id;
    {
        // [Re a_1..a_p][Im a_1..a_p] reduced together
        double v[2 * P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
            v[k] = re[k];
            v[P + k] = im[k];
        }
        const double sum = tc_wave_scatter_sum<2 * P>(v, first, end);
        if (first < end) {
            ex[first] = sum;
            if (dexps)
                dexps[(size_t)2 * P * id + first] = (double)(first < P ? first + 1 : first - P + 1) * sum;
        }
    }
    if (lane == 0) {
        TcNode nd;
        nd.xcom = xc;
        nd.ycom = yc;
        nd.r = rad;
        nd.mass = m;
        nd.s = s;
        nd.e = e;
        nd.child = 0;
        nd.level = l;
        nd.cx = cc.x;
        nd.cy = cc.y;
        nd.rr = rad * rad;
        nodes[id] = nd;
        nodew[id] = make_double4(w, wx, wy, 0.0);
    }
}

// Parent update of upward.cpp:95-218 and upward_e2e (upward-kernels.m4:95-149)
// for internal node `rank`, by one wavefront.  The children's translations run
// in parallel: lane group g (E2E_G lanes: 16 for p <= 16, else 32) takes child
// g of a round, lane l of it the coefficient l + 1.  Every lane runs the
// reference's recurrence for the powers z0^-j itself and keeps the one it
// needs (two dependent operations a step, no LDS round trip), and the binomials
// come from a table in LDS: read from memory inside the sum they were most of
// the kernel's time (one cache round trip per term).  Each child's contribution lands
// in LDS and lanes add them in order c = 0..3, so every coefficient is formed
// by the same operations as a child-by-child loop.
template <int P> constexpr int E2E_G = P <= 16 ? 16 : 32;

// C(l, k) at [k * P + l], k, l < P (0 for k > l): lane l reads consecutive words
template <int P> TC_DEV void e2e_binom(double *s_binom)
{
    for (int i = threadIdx.x; i < P * P; i += blockDim.x)
        s_binom[i] = c_binom[(i % P) * 64 + i / P];
}

// Node data passed between waves of one launch: agent-scope accesses go past
// the XCDs' own L2s, which are not coherent with each other.
template <bool AGENT> TC_DEV unsigned long long node_load_u64(const void *p)
{
    const unsigned long long *q = static_cast<const unsigned long long *>(p);
    return AGENT ? __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *q;
}
template <bool AGENT> TC_DEV double node_load(const double *p)
{
    return __longlong_as_double((long long)node_load_u64<AGENT>(p));
}
template <bool AGENT> TC_DEV void node_store(double *p, double v)
{
    if (AGENT)
        __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), (unsigned long long)__double_as_longlong(v),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        *p = v;
}

// CHAIN: a child was written by this launch; else all by earlier ones (plain,
// cached loads).  SHARED: another wave of this launch may read the node.
template <int P, bool CHAIN, bool SHARED>
TC_DEV void e2e_node(int rank, const int *selfid, const double *box, TcNode *nodes, double4 *nodew, double *exps,
                     double *dexps, double2 (*s_a)[P], double *s_rec, const double *s_binom,
                     double ninv)
{
    constexpr int G = E2E_G<P>, NCH = 64 / G;
    const int lane = tc_lane();
    const int grp = lane / G, gl = lane % G;
    const int cb = 1 + 4 * rank;
    const int id = selfid[rank];

    // the children's records (256 contiguous bytes) and weights (128), a word
    // per lane, and this lane's coefficients: one round of loads.  Level, cell
    // and source range follow from the children's.
    unsigned long long rec = 0;
    if (lane < 48)
        rec = node_load_u64<CHAIN>(lane < 32 ? reinterpret_cast<const double *>(nodes + cb) + lane
                                             : reinterpret_cast<const double *>(nodew + cb) + (lane - 32));
    double2 co[4 / NCH];
#pragma unroll
    for (int q = 0; q < 4 / NCH; ++q) {
        const double *ca = exps + (size_t)2 * P * (cb + q * NCH + grp);
        co[q] = gl < P ? make_double2(node_load<CHAIN>(ca + gl), node_load<CHAIN>(ca + P + gl)) : make_double2(0.0, 0.0);
    }
    if (lane < 48)
        s_rec[lane] = __longlong_as_double((long long)rec);
    tc_wave_sync();
    auto word = [&](int k) { return (unsigned long long)__double_as_longlong(s_rec[k]); };
    const unsigned long long se0 = word(4), se3 = word(8 * 3 + 4), cl0 = word(5), cc0 = word(6);
    const int2 range = make_int2((int)(unsigned)se0, (int)(se3 >> 32));
    const int l = (int)(cl0 >> 32) - 1;
    const int2 cc = make_int2((int)(unsigned)cc0 >> 1, (int)(cc0 >> 32) >> 1);
    const double xmin = box[0], ymin = box[1], ext = box[2];

    double msum = 0, wsum = 0, wxsum = 0, wysum = 0;
    int zcount = 0, nz = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const double w = s_rec[32 + 4 * c];
        msum += s_rec[8 * c + 3];
        wsum += w;
        wxsum += s_rec[32 + 4 * c + 1];
        wysum += s_rec[32 + 4 * c + 2];
        const bool neg = fabs(w) < 1.1e-16;
        zcount += neg;
        if (!neg)
            nz = c;
    }
    // (scaling by 2^-l rounds as dividing by 2^l does)
    const double h = ldexp(ext, -l);
    const double xcp = wsum != 0 ? wxsum / wsum : (xmin + h * (double)cc.x) + 0.5 * h;
    const double ycp = wsum != 0 ? wysum / wsum : (ymin + h * (double)cc.y) + 0.5 * h;
    // radius: lanes c, c + 4, ... take child c; the maximum over the four
    double rr = 0;
    {
        const int c = lane & 3;
        const double rx = xcp - s_rec[8 * c], ry = ycp - s_rec[8 * c + 1];
        const double v = s_rec[8 * c + 2] + sqrt(rx * rx + ry * ry);
        rr = s_rec[32 + 4 * c] != 0 && rr < v ? v : rr;
        double o = tc_xor<1>(rr);
        rr = rr < o ? o : rr;
        o = tc_xor<2>(rr);
        rr = rr < o ? o : rr;
    }
    const double rcap = ldexp((double)1.4143f * ext, -l);
    const double rad = rcap < rr ? rcap : rr;

    double dre = 0, dim = 0;
    if (zcount == 3) {
        if (lane < P) {
            dre = node_load<CHAIN>(exps + (size_t)2 * P * (cb + nz) + lane);
            dim = node_load<CHAIN>(exps + (size_t)2 * P * (cb + nz) + P + lane);
        }
    } else if (zcount < 3) {
        double zr[4 / NCH], zi[4 / NCH], mq[4 / NCH];  // z0^-(gl + 1); the child's mass
        double r1[4 / NCH], i1[4 / NCH], rj[4 / NCH], ij[4 / NCH];
        bool act[4 / NCH], ident[4 / NCH];
#pragma unroll
        for (int q = 0; q < 4 / NCH; ++q) {
            const int c = q * NCH + grp;  // this lane's child
            const double x0 = s_rec[8 * c] - xcp, y0 = s_rec[8 * c + 1] - ycp;
            mq[q] = s_rec[8 * c + 3];
            act[q] = s_rec[32 + 4 * c] != 0;
            ident[q] = x0 == 0 && y0 == 0;
            const double r2z0 = x0 * x0 + y0 * y0;
            zr[q] = rj[q] = r1[q] = x0 / r2z0;
            zi[q] = ij[q] = i1[q] = -y0 / r2z0;
        }
#pragma unroll 4
        for (int j = 1; j < P; ++j) {
#pragma unroll
            for (int q = 0; q < 4 / NCH; ++q) {
                const double rn = rj[q] * r1[q] - ij[q] * i1[q];
                const double in = rj[q] * i1[q] + ij[q] * r1[q];
                rj[q] = rn;
                ij[q] = in;
                zr[q] = j == gl ? rn : zr[q];
                zi[q] = j == gl ? in : zi[q];
            }
        }
#pragma unroll
        for (int q = 0; q < 4 / NCH; ++q)
            if (gl < P)
                s_a[q * NCH + grp][gl] = make_double2(co[q].x * zr[q] - co[q].y * zi[q],
                                                      co[q].x * zi[q] + co[q].y * zr[q]);
        tc_wave_sync();
        double2 res[4 / NCH];
#pragma unroll
        for (int q = 0; q < 4 / NCH; ++q) {
            const double2 *a = s_a[q * NCH + grp];
            double rt = mq[q] * ninv;
            double it = a[0].y;
            rt = rt + a[0].x;
            // lanes past their last term keep their sums by selects, not branches, so that
            // the LDS reads of several terms are in flight (order 24, 10,000 points:
            // chained levels 37 -> 32 us)
            const double *bin = s_binom + (gl < P ? gl : 0);
#pragma unroll(P > 16 ? 8 : 4)
            for (int k = 1; k < P; ++k) {
                const double bk = bin[k * P];
                const double nr = rt + a[k].x * bk, ni = it + a[k].y * bk;
                rt = k <= gl ? nr : rt;
                it = k <= gl ? ni : it;
            }
            const double invz2 = zr[q] * zr[q] + zi[q] * zi[q];
            const double invinv = invz2 != 0 ? 1 / invz2 : 0;
            const double rz = zr[q] * invinv;
            const double iz = -zi[q] * invinv;
            res[q] = make_double2(rt * rz - it * iz, rt * iz + it * rz);
            // z0 = 0 translates by the identity; w = 0 children add nothing
            if (!act[q])
                res[q] = make_double2(0.0, 0.0);
            else if (ident[q])
                res[q] = co[q];
        }
        tc_wave_sync();
#pragma unroll
        for (int q = 0; q < 4 / NCH; ++q)
            if (gl < P)
                s_a[q * NCH + grp][gl] = res[q];
        tc_wave_sync();
        if (lane < P) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const double2 v = s_a[c][lane];
                dre = s_rec[32 + 4 * c] != 0 ? dre + v.x : dre;
                dim = s_rec[32 + 4 * c] != 0 ? dim + v.y : dim;
            }
        }
    }
    if (lane < P) {
        node_store<SHARED>(exps + (size_t)2 * P * id + lane, dre);
        node_store<SHARED>(exps + (size_t)2 * P * id + P + lane, dim);
        if (dexps) {
            dexps[(size_t)2 * P * id + lane] = (double)(lane + 1) * dre;
            dexps[(size_t)2 * P * id + P + lane] = (double)(lane + 1) * dim;
        }
    }
    // the record and weights, a word per lane again
    tc_wave_sync();
    if (lane == 0) {
        auto pair = [](int lo, int hi) {
            return __longlong_as_double((long long)((unsigned)lo | ((unsigned long long)(unsigned)hi << 32)));
        };
        s_rec[0] = xcp;
        s_rec[1] = ycp;
        s_rec[2] = rad;
        s_rec[3] = msum;
        s_rec[4] = pair(range.x, range.y);
        s_rec[5] = pair(cb, l);
        s_rec[6] = pair(cc.x, cc.y);
        s_rec[7] = rad * rad;
        s_rec[8] = wsum;
        s_rec[9] = wxsum;
        s_rec[10] = wysum;
        s_rec[11] = 0.0;
    }
    tc_wave_sync();
    if (lane < 12)
        node_store<SHARED>(lane < 8 ? reinterpret_cast<double *>(nodes + id) + lane
                                    : reinterpret_cast<double *>(nodew + id) + (lane - 8),
                           s_rec[lane]);
    tc_wave_sync();  // s_a and s_rec are rewritten for the wave's next node
}
static_assert(offsetof(TcNode, mass) == 24 && offsetof(TcNode, s) == 32 && offsetof(TcNode, child) == 40 &&
                  offsetof(TcNode, cx) == 48 && offsetof(TcNode, rr) == 56,
              "e2e_node moves records as 8-byte words");

// One wavefront per internal node of one level (ranks r0 .. r1 - 1).
template <int P>
__global__ __launch_bounds__(256) void k_e2e_level(const int *__restrict__ selfid, int r0, int r1,
                                                   const double *__restrict__ box, TcNode *nodes, double4 *nodew,
                                                   double *exps, double *dexps)
{
    __shared__ double s_binom[P * P];
    __shared__ double2 s_a[4][4][P];
    __shared__ double s_rec[4][48];
    e2e_binom<P>(s_binom);
    __syncthreads();
    const int wid = threadIdx.x >> 6, rank = tc_uniform(r0 + (int)blockIdx.x * 4 + wid);
    if (rank < r1)
        e2e_node<P, false, false>(rank, selfid, box, nodes, nodew, exps, dexps, s_a[wid], s_rec[wid], s_binom,
                                  -(1.0 / (double)(tc_lane() % E2E_G<P> + 1)));
}

// The top T internal nodes in one launch, children before parents; those from
// rank tlast on (their level's children come from k_e2e_level) and those whose
// children are all leaves are the starting points, one wave each.  pend[r] =
// (internal children of rank r) << 8 | (of these, not finished yet), parent[r]
// its parent's rank (k_int_nodes).  After a node its wave takes one off the
// parent's count; the wave that takes the last goes on with the parent, the
// others leave, so no wave ever waits for another.  A node's stores have
// completed (vmcnt 0) before its parent's count is taken off.  A level costs
// about 4 us of latency here, but agent-scope traffic makes a node dearer
// (3 ns against 1.5 at 2^24 sources), so levels that fill the GPU go level by
// level and E2E_CHAIN_T nodes or fewer this way.  Upward pass above the leaves,
// with one launch per level above 64 nodes and one workgroup for the levels
// below it (bound by one CU's FP64 rate): 235 -> 146 us at 2^24 sources (order 9),
// 142 -> 90 at 2^23 (order 8), 45 -> 16 at 2^16 (order 12), 71 -> 32 at 10,000
// (order 24).
constexpr int E2E_CHAIN_T = 4096;
// A build whose node bound is at most this is queued without waiting for its census
// (tc_build_tree): bounded by the chained launch, whose waves are started at the
// bound, and by the memory that nodes short of it leave unused.
constexpr long long AHEAD_NODES = 16384;
constexpr size_t AHEAD_BYTES = size_t(48) << 20;
template <int P>
__global__ __launch_bounds__(256) void k_e2e(const int *__restrict__ selfid, const int *__restrict__ parent,
                                             uint32_t *pend, const int *__restrict__ info, int tmax, int tlast,
                                             const double *__restrict__ box,
                                             TcNode *nodes, double4 *nodew, double *exps, double *dexps)
{
    __shared__ double s_binom[P * P];
    __shared__ double2 s_a[4][4][P];
    __shared__ double s_rec[4][48];
    const int wid = threadIdx.x >> 6;
    int rank = tc_uniform((int)(blockIdx.x * 4 + wid));
    const bool start = rank < census_nodes(info, tmax) && (rank >= tlast || (pend[rank] >> 8) == 0);
    if (!__syncthreads_or(start))
        return;
    e2e_binom<P>(s_binom);
    __syncthreads();
    if (!start)
        return;
    const double ninv = -(1.0 / (double)(tc_lane() % E2E_G<P> + 1));  // -1 / (this lane's coefficient index)
    e2e_node<P, false, true>(rank, selfid, box, nodes, nodew, exps, dexps, s_a[wid], s_rec[wid], s_binom, ninv);
    while (rank != 0) {
        const int up = tc_uniform(parent[rank]);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // and no store moves below (a compiler fence here)
        uint32_t left = 0;
        if (tc_lane() == 0)
            left = __hip_atomic_fetch_sub(&pend[up], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffu;
        if (tc_uniform((int)left) != 1)
            break;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        rank = up;
        e2e_node<P, true, true>(rank, selfid, box, nodes, nodew, exps, dexps, s_a[wid], s_rec[wid], s_binom, ninv);
    }
}

// FP32 mirror of the expansions: b_j = a_j / s^j with s = max(r, 1e-30), so
// that the FP32 E2P evaluates sum b_j (s/z)^j with |s/z| < theta (force trees:
// j b_j, the derivative series' coefficients).  Since |a_j| <= sum|v| r^j / j
// and s >= r, scaling the coefficient itself by 1/s j times keeps every
// intermediate bounded (no overflow of s^-j for tiny radii).  Entry p of a
// node's p + 1 records holds the E2P constants (s, Q ln2/2) for potential
// trees (the FP32 E2P works with log2) and (s, Q) for force trees.
template <int P>
__global__ __launch_bounds__(256) void k_exps32(const TcNode *nodes, const double *exps, const int *__restrict__ info,
                                                int tmax, int deriv, float2 *ex32)
{
    // G lanes per node (p + 1 records each), 64 / G nodes per wave
    constexpr int G = P + 1 <= 16 ? 16 : (P + 1 <= 32 ? 32 : 64);
    const int lane = tc_lane();
    const int id = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / G) + lane / G;
    const int k = lane % G;
    if (id > 4 * census_nodes(info, tmax) || k > P)
        return;
    const double r = nodes[id].r;
    const double sc = r > 1e-30 ? r : 1e-30;
    if (k == P) {
        const double q = nodes[id].mass;
        ex32[(size_t)(P + 1) * id + P] = make_float2((float)sc, (float)(deriv ? q : q * 0.34657359027997264));
        return;
    }
    const double *ex = exps + (size_t)2 * P * id;
    // force trees store j b_j, the coefficients of the derivative series
    const double kj = deriv ? (double)(k + 1) : 1.0;
    const double inv = 1.0 / sc;
    double a = kj * ex[k], b = kj * ex[P + k];
    for (int j = 0; j <= k; ++j) {
        a *= inv;
        b *= inv;
    }
    ex32[(size_t)(P + 1) * id + k] = make_float2((float)a, (float)b);
}

// k a_k of every node, for a force tree that was built with FP32 mirrors alone.
__global__ __launch_bounds__(256) void k_deriv(const double *__restrict__ exps, size_t total, int p,
                                               double *__restrict__ dexps)
{
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256)
        dexps[i] = (double)((int)(i % (size_t)p) + 1) * exps[i];
}

int tiles_of(int n, int t) { return (n + t - 1) / t; }

}  // namespace

// ================================================================== host side

void tc_fill_u32(uint32_t *p, uint32_t v, size_t n, hipStream_t st)
{
    if (!n)
        return;
    const int grid = (int)std::min<size_t>((n + 255) / 256, 4096);
    k_fill_u32<<<grid, 256, 0, st>>>(p, v, n);
    TC_HIP(hipGetLastError());
}

void tc_upload_binomials(hipStream_t st)
{
    std::vector<double> tab(64 * 64, 0.0);
    for (int n = 0; n < 64; ++n)
        for (int k = 0; k <= n; ++k) {
            unsigned __int128 r = 1;
            const int kk = k < n - k ? k : n - k;
            for (int i = 1; i <= kk; ++i)
                r = r * (unsigned __int128)(n - kk + i) / (unsigned __int128)i;
            tab[n * 64 + k] = (double)r;
        }
    TC_HIP(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_binom), tab.data(), sizeof(double) * tab.size(), 0,
                                  hipMemcpyHostToDevice, st));
    TC_HIP(hipStreamSynchronize(st));
}

static const uint32_t *tc_bbox_bad_flag(TcScratch &ws, int n)
{
    const int np = std::max(1, std::min(1024, tiles_of(n, 256 * 8)));
    return reinterpret_cast<const uint32_t *>(ws.bbox_part.as<double4>() + np);
}

// A set's device memory for a sort with one-launch passes (small: one-workgroup
// sort): np bounding-box partials, the non-finite flag where tc_bbox_bad_flag finds
// it, per-workgroup flags after it.
static SortSet sort_set(const double *x, const double *y, const double *v, int n, double *box, uint32_t *keys,
                        uint32_t *perm, double4 *records, TcScratch &ws, bool small)
{
    SortSet t = {};
    t.x = x;
    t.y = y;
    t.v = v;
    t.n = n;
    t.box = box;
    t.keys = keys;
    t.perm = perm;
    t.np = std::max(1, std::min(1024, tiles_of(n, 256 * 8)));
    if (small) {
        ws.bbox_part.reserve(sizeof(double4) * (size_t)t.np + 256);
        t.bad = const_cast<uint32_t *>(tc_bbox_bad_flag(ws, n));
        return t;
    }
    ws.bbox_part.reserve(sizeof(double4) * (size_t)t.np + 256 + sizeof(uint32_t) * (size_t)t.np);
    t.part = ws.bbox_part.as<double4>();
    t.bad = const_cast<uint32_t *>(tc_bbox_bad_flag(ws, n));
    t.pbad = t.bad + 64;
    t.ntiles = tiles_of(n, RS_NT * rs_items(n));
    if (lb_words(t.ntiles) > (size_t)INT_MAX)
        throw TcError(-3, "tc_sort_points: too many points");
    // the counts of a sort with records lie where the sorted records come later
    if (records && sizeof(uint32_t) * lb_words(t.ntiles) <= sizeof(double4) * (size_t)n) {
        t.lb = reinterpret_cast<uint32_t *>(records);
    } else {
        ws.hist.reserve(sizeof(uint32_t) * lb_words(t.ntiles));
        t.lb = ws.hist.as<uint32_t>();
    }
    ws.k2.reserve(sizeof(uint32_t) * (size_t)n);
    ws.v2.reserve(sizeof(uint32_t) * (size_t)n);
    t.k2 = ws.k2.as<uint32_t>();
    t.v2 = ws.v2.as<uint32_t>();
    if (records) {
        ws.packed.reserve(sizeof(double4) * (size_t)n);
        t.packed = ws.packed.as<double4>();
    }
    // at most KH_TILE_MAX points a step, at least KH_TILE_MIN, about one step per CU
    t.kstep = std::min(KH_TILE_MAX, std::max(KH_TILE_MIN, tiles_of(tiles_of(n, 1024), 256) * 1024));
    t.kgrid = std::min(tiles_of(n, t.kstep), KH_GRID);
    return t;
}

// Sorts one or two sets (the second with n = 0 for one); both small or neither.
// src_out: the first set's sorted records; tp: the first set's topology (small
// sorts only).
static void sort_sets(const SortSets &t, double4 *src_out, const SmallTopo &tp, hipStream_t st, const hipEvent_t *ev)
{
    const int sets = t.s[1].n > 0 ? 2 : 1;
    if (t.s[0].n <= SS_N) {
        small_items(std::max(t.s[0].n, t.s[1].n), [&](auto it) {
            k_sort_small<decltype(it)::value><<<sets, SS_NT, 0, st>>>(t, src_out, tp);
        });
        TC_HIP(hipGetLastError());
        if (ev) {
            // one kernel does keys and sort: both boundaries fall after it
            TC_HIP(hipEventRecord(ev[0], st));
            TC_HIP(hipEventRecord(ev[1], st));
        }
        return;
    }
    // the box, the keys with all passes' digit totals, then one launch per pass
    const int ntiles = t.s[0].ntiles + t.s[1].ntiles;
    k_bbox_partial<<<t.s[0].np + t.s[1].np, 256, 0, st>>>(t, (int)lb_words(t.s[0].ntiles),
                                                          sets == 2 ? (int)lb_words(t.s[1].ntiles) : 0);
    k_keys_hist<<<t.s[0].kgrid + t.s[1].kgrid, 256, 0, st>>>(t);
    TC_HIP(hipGetLastError());
    if (ev)
        TC_HIP(hipEventRecord(ev[0], st));
    // (two sets are sorted together only where both have the fewest keys per thread)
    const int items = rs_items(t.s[0].n);
    const auto pass_kernel = items == 5 ? k_rs_pass_lb<5> : items == 8 ? k_rs_pass_lb<8> : k_rs_pass_lb<15>;
    for (int pass = 0; pass < RS_PASSES; ++pass)
        pass_kernel<<<ntiles, RS_NT, 0, st>>>(t, pass);
    if (src_out)
        k_gather_src<<<tiles_of(t.s[0].n, 256), 256, 0, st>>>(t.s[0].packed, t.s[0].perm, t.s[0].n, src_out);
    TC_HIP(hipGetLastError());
    if (ev)
        TC_HIP(hipEventRecord(ev[1], st));
}

void tc_morton_sort(const double *x, const double *y, int n, double *box_d, uint32_t *keys, uint32_t *perm,
                    TcScratch &ws, hipStream_t st)
{
    SortSets t = {};
    // (any non-null strengths make Morton keys; without records they are not read)
    t.s[0] = sort_set(x, y, x, n, box_d, keys, perm, nullptr, ws, n <= SS_N);
    sort_sets(t, nullptr, SmallTopo{}, st, nullptr);
}

// Targets' buffers in ws: keys, permutation, and the box after the source box's place.
static SortSet target_set(const double *xt, const double *yt, int m, TcScratch &ws, bool small)
{
    ws.tkeys.reserve(sizeof(uint32_t) * (size_t)m + 64);
    ws.tperm.reserve(sizeof(uint32_t) * (size_t)m + 64);
    ws.info.reserve(sizeof(int) * 32 + sizeof(double) * 4);
    return sort_set(xt, yt, nullptr, m, reinterpret_cast<double *>(ws.info.as<char>() + 128), ws.tkeys.as<uint32_t>(),
                    ws.tperm.as<uint32_t>(), nullptr, ws, small);
}

// Sources and targets up to here in total go through one set of launches; beyond, the
// GPU is filled by either, and the targets' sort runs beside the build on a stream of
// its own.
constexpr int SORT_JOINT_MAX = 1 << 20;
static_assert(rs_items(SORT_JOINT_MAX) == 5, "one tile size for both sets");
bool tc_sorts_jointly(int n, int m)
{
    if (n <= 0 || m <= 0)
        return false;
    return n <= SS_N ? m <= SS_N : m > SS_N && (long long)n + m <= SORT_JOINT_MAX;
}

// info, tmax: the tree's internal nodes as the kernels read them (at most tmax);
// starts: its level starts, or null where the host does not have them yet (all
// levels then go in the chained launch).
template <int P>
static void upward_launch(TcTree &t, const uint32_t *child, const int2 *se, const int *lev, const int2 *cell,
                          const int *parent, uint32_t *pend, bool fp32, bool deriv, const int *info, int tmax,
                          const int *starts, hipStream_t st)
{
    const double *box = t.box_d.as<double>();
    double *dexps = t.has_deriv ? t.dexps.as<double>() : nullptr;
    const int nn = 1 + 4 * tmax;
    k_leaf_upward<P><<<tiles_of(nn, 4), 256, 0, st>>>(child, se, lev, cell, t.src.as<double4>(), box, info, tmax,
                                                      t.nodes.as<TcNode>(), t.exps.as<double>(), dexps,
                                                      t.nodew.as<double4>(), fp32 ? t.src32.as<float4>() : nullptr);
    TC_HIP(hipGetLastError());
    // levels lt and below one launch each, the levels above in one
    int top = tmax, last = INT_MAX;
    if (starts) {
        int lt = TC_LMAX;
        while (starts[lt] > E2E_CHAIN_T)
            --lt;
        for (int L = TC_LMAX - 1; L >= lt; --L) {
            const int r0 = starts[L], r1 = starts[L + 1];
            if (r1 > r0) {
                k_e2e_level<P><<<tiles_of(r1 - r0, 4), 256, 0, st>>>(t.selfid.as<int>(), r0, r1, box,
                                                                      t.nodes.as<TcNode>(), t.nodew.as<double4>(),
                                                                      t.exps.as<double>(), dexps);
                TC_HIP(hipGetLastError());
            }
        }
        top = starts[lt];
        if (lt < TC_LMAX)
            last = starts[lt - 1];
    }
    if (top > 0) {
        k_e2e<P><<<tiles_of(top, 4), 256, 0, st>>>(t.selfid.as<int>(), parent, pend, info, top, last, box,
                                                   t.nodes.as<TcNode>(), t.nodew.as<double4>(), t.exps.as<double>(),
                                                   dexps);
        TC_HIP(hipGetLastError());
    }
    if (fp32) {
        constexpr int per_wave = P + 1 <= 16 ? 4 : (P + 1 <= 32 ? 2 : 1);
        k_exps32<P><<<tiles_of(nn, 4 * per_wave), 256, 0, st>>>(t.nodes.as<TcNode>(), t.exps.as<double>(), info, tmax,
                                                                 deriv ? 1 : 0, t.exps32.as<float2>());
        TC_HIP(hipGetLastError());
    }
}

// Most internal nodes that n sources with this leaf capacity can have: the
// cells of a level are disjoint and hold more than leafcap sources each.
static long long internal_bound(int n, int leafcap)
{
    const long long per_level = (long long)n / ((long long)leafcap + 1);
    long long t = 0;
    for (int L = 0; L < TC_LMAX; ++L)
        t += std::min(per_level, 1ll << (2 * L));
    return t;
}

void tc_build_tree(TcTree &t, const double *x, const double *y, const double *v, int n, int leafcap, int order,
                   bool fp32, bool deriv, TcScratch &ws, hipStream_t st, const hipEvent_t *ev,
                   const std::function<void()> *at_census, TcJointTargets *targets)
{
    if (n <= 0)
        throw TcError(-3, "tc_build_tree: no sources");
    if (leafcap < 1 || leafcap > TC_MAX_LEAF)
        throw TcError(-3, "tc_build_tree: leaf capacity must be in [1, 2^30]");
    if (n >= (1 << 30))
        throw TcError(-3, "tc_build_tree: at most 2^30 - 1 sources per tree");
    if (!tc_order_supported(order))
        throw TcError(-3, "tc_build_tree: unsupported expansion order " + std::to_string(order));
    t.n = n;
    t.order = order;
    t.leafcap = leafcap;
    t.has_fp32 = fp32;
    t.deriv32 = fp32 && deriv;
    t.has_deriv = !fp32 && deriv;
    t.box_d.reserve(sizeof(double) * 4);
    t.keys.reserve(sizeof(uint32_t) * (size_t)n);
    t.perm.reserve(sizeof(uint32_t) * (size_t)n);
    t.src.reserve(sizeof(double4) * (size_t)n);
    if (fp32)
        t.src32.reserve(sizeof(float4) * (size_t)n);

    double *box = t.box_d.as<double>();
    uint32_t *keys = t.keys.as<uint32_t>(), *perm = t.perm.as<uint32_t>();
    const bool small = n <= SS_N;
    SortSets sets = {};
    sets.s[0] = sort_set(x, y, v, n, box, keys, perm, t.src.as<double4>(), ws, small);
    const uint32_t *tbad = nullptr;
    if (targets) {
        sets.s[1] = target_set(targets->x, targets->y, targets->m, *targets->ws, small);
        tbad = sets.s[1].bad;
    }
    ws.info.reserve(sizeof(int) * 32 + sizeof(double) * 4);
    int *info = ws.info.as<int>();
    static_assert(INFO_BYTES <= sizeof(int) * 32 && INFO_BYTES <= TcScratch::PINNED_BYTES, "census record size");
    char *hp = static_cast<char *>(ws.host_pinned());
    int *hrec = reinterpret_cast<int *>(hp);

    // Where the bound on the node count fits a modest buffer, the rest of the
    // build is queued behind the census at that bound (its kernels read the count on the
    // device), and the host waits for the record while they run: queued after the
    // readback instead, they start one host round trip and launch after the
    // other with the GPU idle in between. 4 to 5% of a 0.3 to 0.5 ms
    // solve (65,536-point FP64 potential 288 -> 278 us).
    const size_t per_node = sizeof(TcNode) + sizeof(double4) + 24 + 16 * (size_t)order * (t.has_deriv ? 2 : 1) +
                            (fp32 ? 8 * ((size_t)order + 1) : 0);
    const long long bound = internal_bound(n, leafcap);
    const bool ahead = !t.nodes.arena && bound <= AHEAD_NODES && (1 + 4 * (size_t)bound) * per_node <= AHEAD_BYTES;
    const bool topo_small = ahead && small && bound <= SMALL_TOPO_T;

    int T = (int)std::min<long long>(bound, INT_MAX / 8), hinfo[TC_LMAX + 3];
    uint32_t *child = nullptr, *pend = nullptr;
    int2 *se = nullptr, *cell = nullptr;
    int *lev = nullptr, *istart = nullptr, *ilevel = nullptr;
    // buffers of a tree of at most T internal nodes
    auto reserve_nodes = [&] {
        const size_t nn = 1 + 4 * (size_t)T;
        t.nodes.reserve(sizeof(TcNode) * nn);
        t.exps.reserve(sizeof(double) * 2 * (size_t)order * nn);
        if (t.has_deriv)
            t.dexps.reserve(sizeof(double) * 2 * (size_t)order * nn);
        t.nodew.reserve(sizeof(double4) * nn);
        t.selfid.reserve(sizeof(int) * (size_t)(T + 1));
        if (fp32)
            t.exps32.reserve(sizeof(float2) * (size_t)(order + 1) * nn);
        ws.istart.reserve(sizeof(int) * 2 * (size_t)(T + 1));
        istart = ws.istart.as<int>();
        pend = ws.istart.as<uint32_t>() + T + 1;
        ws.ilevel.reserve(sizeof(int) * (size_t)(T + 1));
        ilevel = ws.ilevel.as<int>();
        // per-node topology scratch: child | se | level | cell
        ws.ints.reserve(sizeof(int) * nn * 6 + 64);
        child = ws.ints.as<uint32_t>();
        se = reinterpret_cast<int2 *>(child + ((nn + 1) & ~size_t(1)));
        lev = reinterpret_cast<int *>(se + nn);
        cell = reinterpret_cast<int2 *>(lev + ((nn + 1) & ~size_t(1)));
    };
    SmallTopo tp = {};
    if (ahead)
        reserve_nodes();
    if (topo_small) {
        tp.cap = leafcap;
        tp.tmax = std::max(1, T);
        tp.info = info;
        tp.hinfo = hrec;
        tp.selfid = t.selfid.as<int>();
        tp.parent = ilevel;
        tp.pend = pend;
        tp.child = child;
        tp.se = se;
        tp.level = lev;
        tp.cell = cell;
    }
    sort_sets(sets, t.src.as<double4>(), tp, st, ev);

    // census of internal cells
    const bool few = n <= TB_SMALL_N;
    const int nblk = tiles_of(n, 256 * (few ? TB_IT_SMALL : TB_IT));
    const int stride = (nblk + 3) & ~3;
    uint32_t *cnt = nullptr, *offs = nullptr;
    if (!topo_small) {
        ws.part.reserve(sizeof(uint32_t) * (size_t)2 * TC_LMAX * stride);
        cnt = ws.part.as<uint32_t>();
        offs = cnt + (size_t)TC_LMAX * stride;
        if (few)
            k_int_count<TB_IT_SMALL><<<nblk, 256, 0, st>>>(keys, n, leafcap, cnt, stride);
        else
            k_int_count<TB_IT><<<nblk, 256, 0, st>>>(keys, n, leafcap, cnt, stride);
        k_census<<<1, SCAN_NT, 0, st>>>(cnt, offs, nblk, stride, sets.s[0].bad, tbad, box, info, hrec);
        TC_HIP(hipGetLastError());
    }
    if (ahead)
        TC_HIP(hipEventRecord(ws.census_event(), st));
    if (at_census)
        (*at_census)();  // work queued elsewhere fills the GPU while the host waits
    const int *starts = nullptr;
    auto census = [&] {
        if (ahead)
            TC_HIP(hipEventSynchronize(ws.census_event()));
        else
            TC_HIP(hipStreamSynchronize(st));
        std::memcpy(hinfo, hp, sizeof(hinfo));
        std::memcpy(t.box, hp + sizeof(int) * INFO_BOX, sizeof(t.box));
        if (hinfo[TC_LMAX + 1]) {
            TC_HIP(hipStreamSynchronize(st));  // no kernel of a failed build outlives the call
            if (hinfo[TC_LMAX + 1] & 2)
                throw TcError(-9, "treecode: the source sort did not complete (a radix pass timed out)");
            throw TcError(-4, "treecode: non-finite source coordinate");
        }
        for (int L = 0; L <= TC_LMAX; ++L)
            t.level_start[L] = hinfo[L];
        t.level_start[TC_LMAX + 1] = hinfo[TC_LMAX];
        t.ninternal = hinfo[TC_LMAX];
        t.nnodes = 1 + 4 * t.ninternal;
        if (targets)
            targets->bad = (uint32_t)hinfo[TC_LMAX + 2];
    };
    if (!ahead) {
        census();
        T = t.ninternal;
        starts = t.level_start;
        reserve_nodes();
    }
    if (!topo_small) {
        if (T > 0 && few)
            k_int_emit<TB_IT_SMALL><<<nblk, 256, 0, st>>>(keys, n, leafcap, offs, stride, T, istart, ilevel);
        else if (T > 0)
            k_int_emit<TB_IT><<<nblk, 256, 0, st>>>(keys, n, leafcap, offs, stride, T, istart, ilevel);
        const bool by_wave = T <= NODES_WAVE_T;
        const auto nodes_kernel = by_wave ? k_int_nodes<64> : k_int_nodes<16>;
        nodes_kernel<<<std::max(1, tiles_of(T, by_wave ? 4 : 16)), 256, 0, st>>>(
            keys, n, leafcap, istart, ilevel, info, T, t.selfid.as<int>(), pend, child, se, lev, cell);
        TC_HIP(hipGetLastError());
    }
    if (ev)
        TC_HIP(hipEventRecord(ev[2], st));

    switch (order) {
#define TC_CASE(P) \
    case P: upward_launch<P>(t, child, se, lev, cell, ilevel, pend, fp32, deriv, info, T, starts, st); break;
        TC_ORDERS(TC_CASE)
#undef TC_CASE
    }
    if (ev)
        TC_HIP(hipEventRecord(ev[3], st));
    if (ahead)
        census();
}

void tc_tree_deriv(TcTree &t, hipStream_t st)
{
    if (t.has_deriv)
        return;
    const size_t total = 2 * (size_t)t.order * t.nnodes;
    t.dexps.reserve(sizeof(double) * total);
    k_deriv<<<(int)std::min<size_t>((total + 255) / 256, 4096), 256, 0, st>>>(t.exps.as<double>(), total, t.order,
                                                                           t.dexps.as<double>());
    TC_HIP(hipGetLastError());
    t.has_deriv = true;
}

const uint32_t *tc_targets_bad_flag(TcScratch &ws, int m) { return tc_bbox_bad_flag(ws, m); }

TcSortDesc tc_sort_targets_desc(const double *xt, const double *yt, int m, TcScratch &ws)
{
    if (m < 1 || m > SS_N)
        throw TcError(-3, "tc_sort_targets_desc: 1 to 16384 targets");
    // the buffers and places tc_sort_targets uses for m targets
    const SortSet t = target_set(xt, yt, m, ws, true);
    TcSortDesc d;
    d.x = xt;
    d.y = yt;
    d.box = t.box;
    d.bad = t.bad;
    d.keys = t.keys;
    d.perm = t.perm;
    d.n = m;
    d.pad = 0;
    return d;
}

void tc_sort_targets_batch(const TcSortDesc *desc_dev, int k, int mmax, hipStream_t st)
{
    if (k <= 0)
        return;
    small_items(mmax, [&](auto it) { k_sort_small_batch<decltype(it)::value><<<k, SS_NT, 0, st>>>(desc_dev); });
    TC_HIP(hipGetLastError());
}

void tc_sort_targets(const double *xt, const double *yt, int m, TcScratch &ws, hipStream_t st)
{
    SortSets t = {};
    t.s[0] = target_set(xt, yt, m, ws, m <= SS_N);
    sort_sets(t, nullptr, SmallTopo{}, st, nullptr);
}
