// tc.hip -- triangle counting (HornetsNest TriangleCounting2).
//
// Reference: TriangleCounting2::run -> forAllAdjUnions
// (primitives/Operator++.i.cuh:369-475) bins every stored edge by estimated
// work into 2,048 bins with 64-bit atomics, copies the bin sizes to the host,
// and launches up to 39 merge-path / binary-search intersection kernels
// (:97-246), each followed by a device sync; the operator
// (hornetsnest/src/Static/TriangleCounting/triangle2.cu:75-124) skips
// src == dst and deg(src) < 2, intersects N(u) with N(v) where u is the
// endpoint with the smaller degree (ties -> the destination), and credits u.
// The driver stores the DIRECTED_BY_DEGREE orientation
// (hornetsnest/test/TriangleTest2.cu:86-87, xlib/src/Graph/GraphStd.cpp:247-304),
// so the sum is the triangle count.
//
// Here an edge is intersected where its longer list is: the owner of an edge is
// the endpoint with the longer list, a workgroup puts the owner's list into LDS
// once, and then walks the shorter lists of the owner's edges, one LDS test per
// entry and no search.  Over an R-MAT s22 orientation (64 M edges) that is
// 11.8 G tests of streamed entries; binary searches and 64-entry windows of both
// lists, one edge at a time, took 75 ms for them; here 7.4.
//   * The LDS set is exact: the most frequent vertices (hubs, up to 65,535 of
//     them) have 16-bit codes and one bit each in an 8 KB bitmap; the others are
//     hashed.  A list is two rows, its hubs' codes and the others' ids, each
//     16-byte aligned and padded, so a lane loads eight codes at once and a test
//     is one LDS word and a bit-field extract.  Skewed graphs put nearly all
//     entries on hubs (R-MAT s22: 96 % of the tests), and an owner that is a hub
//     of a degree orientation has nothing but hubs in its list, so that its
//     other tests are skipped altogether.
//   * The orientation keeps (u, v) iff (deg u, u) < (deg v, v): one pass over the
//     stored entries that compacts every row into its own place (the order
//     within a row does not matter to an LDS set).
//   * An owner's edges: on simple symmetric storage its stored row, of which it
//     takes the neighbours with shorter lists.  Otherwise (stored graphs, repeated
//     entries, symmetry not known) its own list, and the sources of the edges
//     whose longer list is the destination's, grouped by it first.
//   * Owners are cut into tasks of up to TC_CAND candidates, which resident
//     workgroups take from a ticket.  Edges between lists of at most TC_SMALL
//     entries are compared in registers by one thread per source.
//   * The count of an edge is credited to the shorter list's vertex with one
//     atomic; the total is summed per workgroup.
#include "graph.hpp"
#include "prims.hpp"

namespace hn {
namespace {

constexpr int TC_G = 8;                        // entries per group: 16 bytes of hub codes, 32 of ids
constexpr uint32_t TC_HUBS = 65535;            // hubs at most
constexpr uint32_t TC_PAD16 = 0xFFFF;          // fills the last group of a row of codes: a bit never set
constexpr uint32_t TC_PAD = 0xFFFFFFFFu;       // ... of a row of ids
constexpr uint32_t TC_ID = 0x80000000u;        // (in a vertex's code) no hub: TC_ID | id
constexpr int TC_BINS = 4096;
constexpr uint32_t TC_SMALL = 16;              // lists up to this long are compared in registers,
constexpr uint32_t TC_SMALL_GROUPED = 32;      // up to this where there are many and owners' edges are grouped
constexpr uint32_t TC_CAND = 1024;             // candidates per task
constexpr int TC_STEP = 2 * BLOCK;             // ... listed at a time
constexpr uint32_t TC_TAIL = 256;              // ids hashed at a time
constexpr uint32_t TC_HASH = 2 * TC_TAIL;
constexpr uint32_t TC_WIDE_HASH = (TC_HUBS + 1) / 32, TC_WIDE_TAIL = TC_WIDE_HASH / 2;   // ... in the bits' place
// Stored rows with more ids are searched, as they are sorted, and not hashed: hashing
// them goes over all candidates once per table, which is quadratic (all stored entries of
// R-MAT s20: 930 ms, a star of four million leaves: 1 s; so: 56 and 0.8 ms.  R-MAT s18 and
// s20, searched from one table less on: 6.7 and 57 ms, from two more on: 8.1 and 64).  The
// lists of an orientation are not whole rows, and long ones of ids take more than 65,535
// vertices of a like degree: they are hashed, one table of 1,024 after the other (cliques
// of 700, in tables of 256: 18.3 ms, 3.3 so; of 5,000: 0.89 s).
constexpr uint32_t TC_SEARCH = TC_TAIL + 2 * TC_WIDE_TAIL;
constexpr int TC_TEAM = 8;                     // lanes per shorter list
constexpr int TC_DEPTH = 4;                    // groups per lane in flight (2 and 8: 3 and 2 % slower on R-MAT s22)
constexpr int TC_ORDER = 32;                   // classes of list lengths that a step is sorted by
constexpr int TC_IPT = 2;                      // groups per lane of the passes over rows
constexpr int TC_TILE = BLOCK * TC_IPT;

// A list: its rows' place in groups, the hubs' and the others' number.
struct __attribute__((aligned(16))) TcRow {
    uint32_t base;
    uint32_t pad;
    uint32_t n16;
    uint32_t n32;
    __device__ __forceinline__ uint32_t len() const { return n16 + n32; }
};

// Atomics on one address take 10 ns each, whoever makes them: the sums and the
// tasks' tickets are spread over lines of their own.
constexpr int TC_SUMS = 32, TC_LANES = 8;
struct alignas(128) TcSum {
    unsigned long long v;
};
struct alignas(128) TcTicket {
    uint32_t v;
};
struct TcCtl {
    TcSum total[TC_SUMS];
    TcTicket ticket[TC_LANES];
    uint64_t owned;      // grouped edges, and the number of tasks << 32
    uint32_t cut;        // bins from this one on are hubs
    uint32_t hubs;
    uint32_t repeats;    // some row stores an entry twice
};

// monotone in d: exponent and seven bits of mantissa
__device__ __forceinline__ uint32_t tc_bin(uint32_t d) {
    if (d == 0) return 0;
    const int e = 31 - __clz((int)d);
    return (uint32_t)e * 128u + (uint32_t)(((uint64_t)d << 7 >> e) & 127u);
}

// ---- hubs: the weights' histogram, the bin from which at most TC_HUBS vertices
// lie, and every vertex's code
__global__ __launch_bounds__(BLOCK) void tc_hist_kernel(int64_t nv, const uint32_t* __restrict__ weight,
                                                        uint32_t* __restrict__ hist) {
    __shared__ uint32_t h[TC_BINS];
    for (int i = threadIdx.x; i < TC_BINS; i += BLOCK) h[i] = 0;
    __syncthreads();
    constexpr int K = 8;   // loads in flight (one: 45 us for 16 M vertices, 22 so)
    for (int64_t b = (int64_t)blockIdx.x * (K * BLOCK); b < nv; b += (int64_t)gridDim.x * (K * BLOCK)) {
        uint32_t w[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int64_t v = b + k * BLOCK + threadIdx.x;
            w[k] = v < nv ? weight[v] : 0u;
        }
#pragma unroll
        for (int k = 0; k < K; k++)
            if (w[k] > 1) atomicAdd(&h[tc_bin(w[k])], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < TC_BINS; i += BLOCK)
        if (h[i]) atomicAdd(hist + i, h[i]);
}

__global__ __launch_bounds__(BLOCK) void tc_cut_kernel(const uint32_t* __restrict__ hist, TcCtl* __restrict__ ctl) {
    __shared__ uint32_t sc[NWAVES + 1];
    __shared__ uint32_t cut;
    if (threadIdx.x == 0) cut = TC_BINS;
    __syncthreads();
    constexpr int K = TC_BINS / BLOCK;
    // thread t sums bins from the top: t * K .. t * K + K - 1 below TC_BINS
    uint32_t x[K], sum = 0;
    for (int k = 0; k < K; k++) {
        x[k] = hist[TC_BINS - 1 - (threadIdx.x * K + k)];
        sum += x[k];
    }
    uint32_t tot;
    uint32_t run = block_exclusive_scan(sum, sc, &tot), mine = TC_BINS;
    for (int k = 0; k < K; k++) {
        run += x[k];
        if (run <= TC_HUBS) mine = (uint32_t)(TC_BINS - 1 - (threadIdx.x * K + k));
    }
    if (mine < TC_BINS) atomicMin(&cut, mine);
    __syncthreads();
    if (threadIdx.x == 0) ctl->cut = cut;
}

struct HubIn {
    const uint32_t* weight;
    const TcCtl* ctl;
    __device__ __forceinline__ uint32_t operator()(int64_t v) const {
        const uint32_t w = weight[v];
        return w > 1 && tc_bin(w) >= ctl->cut ? 1u : 0u;
    }
};
// (weight, code) side by side: the orientation looks up both of every entry; and a bit
// per vertex, for the passes that need a hub's code only (a wave has a word of `hubs`)
struct HubOut {
    const uint32_t* weight;
    uint2* wc;
    uint32_t* hub;
    uint64_t* hubs;
    __device__ __forceinline__ void operator()(int64_t v, uint32_t ex, uint32_t is) const {
        const uint64_t any = __ballot(is != 0);
        if (v % WAVE == 0) hubs[v / WAVE] = any;
        wc[v] = make_uint2(weight[v], is ? ex : (TC_ID | (uint32_t)v));
        if (is) hub[ex] = (uint32_t)v;
    }
};

// Where every vertex can have a bit there is nothing to choose: codes are the
// ids.  One launch in place of six (weights, histogram, cut and codes), 110 us of
// the 590 that a stored graph of 6 K vertices and 100 K entries took.
__global__ void tc_all_hubs_kernel(int64_t nv, const hn_vrec* __restrict__ rec, uint2* __restrict__ wc,
                                   uint32_t* __restrict__ hub, TcCtl* __restrict__ ctl) {
    const int64_t v = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (v == 0) ctl->hubs = (uint32_t)nv;
    if (v >= nv) return;
    wc[v] = make_uint2((uint32_t)rec[v].deg, (uint32_t)v);
    hub[v] = (uint32_t)v;
}

// ---- rows
// groups of the stored rows, prefix summed: a row's place (its list is no
// longer), and the partition for the pass over the entries
struct StoredGroupsIn {
    const hn_vrec* rec;
    __device__ __forceinline__ uint32_t operator()(int64_t v) const { return ((uint32_t)rec[v].deg + TC_G - 1) / TC_G; }
};
// body(v, first, k) for every k of a lane's [first, last): one lane's long range by all
// lanes that are here, those without a range too (a star of four million leaves: its 4,096 tasks by one lane 128 us).
template <typename Body>
__device__ __forceinline__ void tc_spread(uint32_t v, uint32_t first, uint32_t last, Body body) {
    constexpr uint32_t OWN = 16;
    const uint32_t n = last > first ? last - first : 0u;
    if (n <= OWN)
        for (uint32_t k = 0; k < n; k++) body(v, first, first + k);
    uint64_t more = __ballot(n > OWN);
    const uint64_t here = __ballot(true);
    const uint32_t lanes = (uint32_t)__popcll(here), rank = (uint32_t)__popcll(here & lanemask_lt());
    for (; more; more &= more - 1) {
        const int from = __ffsll((unsigned long long)more) - 1;
        const uint32_t w = __shfl(v, from, WAVE), a = __shfl(first, from, WAVE), b = __shfl(last, from, WAVE);
        for (uint32_t k = a + rank; k < b; k += lanes) body(w, a, k);
    }
}
__device__ __forceinline__ void tc_tiles(uint32_t* __restrict__ tile_lo, int64_t v, uint32_t ex, uint32_t x) {
    auto tile = [](uint64_t g) { return (uint32_t)((g + TC_TILE - 1) / TC_TILE); };   // the first that starts at g or later
    tc_spread((uint32_t)v, tile(ex), tile((uint64_t)ex + x), [&](uint32_t w, uint32_t, uint32_t t) { tile_lo[t] = w; });
}
// weight, where given: the degrees, from records that were just read
// (a wave has the 64 vertices of one word of `some`)
struct StoredGroupsOut {
    const hn_vrec* rec;
    TcRow* row;
    uint32_t* P;
    uint32_t* tile_lo;
    uint32_t* weight;
    uint64_t* some;
    __device__ __forceinline__ void operator()(int64_t v, uint32_t ex, uint32_t x) const {
        const uint64_t any = __ballot(x != 0);
        if (v % WAVE == 0) some[v / WAVE] = any;
        if (weight) weight[v] = (uint32_t)rec[v].deg;
        row[v] = TcRow{ex, 0u, 0u, 0u};
        P[v] = ex;
        tc_tiles(tile_lo, v, ex, x);
    }
};

using TcLb = LbShared<TC_IPT, uint32_t, uint32_t>;

// A tile's rows staged and its groups located: group j of the lane is the k-th
// of row seg (seg < 0 past the end).
struct TcLoc {
    int64_t seg[TC_IPT];
    uint32_t k[TC_IPT];
};
template <typename BaseFn>
__device__ __forceinline__ TcLoc tc_locate(const uint32_t* __restrict__ P, int64_t nv, uint32_t total,
                                           const uint32_t* __restrict__ tile_lo, int64_t t, int64_t ntiles, TcLb& sh,
                                           BaseFn base, uint32_t (&b)[TC_IPT]) {
    const int64_t lo = tile_lo[t], hi = t + 1 < ntiles ? (int64_t)tile_lo[t + 1] : nv - 1;
    const int64_t span = hi - lo + 1;
    const bool staged = span <= TcLb::CAP;
    if (staged)
        for (int i = threadIdx.x; i < (int)span; i += BLOCK) {
            sh.pref[i] = P[lo + i];
            sh.base[i] = base(lo + i);
        }
    __syncthreads();
    TcLoc c;
#pragma unroll
    for (int j = 0; j < TC_IPT; j++) {
        const int64_t w = t * TC_TILE + (int64_t)j * BLOCK + threadIdx.x;
        c.seg[j] = -1;
        c.k[j] = 0;
        b[j] = 0;
        if (w < (int64_t)total) {
            if (staged) {
                const int s = lb_locate(sh, (int)span, w);
                c.seg[j] = lo + s;
                c.k[j] = (uint32_t)w - sh.pref[s];
                b[j] = sh.base[s];
            } else {
                const int64_t s = upper_bound_m1<int64_t>(P, lo, hi + 1, w);
                c.seg[j] = s;
                c.k[j] = (uint32_t)w - P[s];
                b[j] = base(s);
            }
        }
    }
    return c;
}

// How often a vertex is an entry, from every `step`-th tile of the stored rows
// (any choice of hubs gives the same counts).  Bound by the atomics on the most
// frequent one, 10 ns each: a quarter of a million to a million entries are looked
// at (all 2.8 M of an R-MAT s18 orientation took 660 us, 73 so), and a wave adds the
// entries equal to its first one together (a star of four million leaves: 1538 us without,
// 34 so).
__global__ __launch_bounds__(BLOCK) void tc_weight_freq_kernel(int64_t nv, const uint32_t* __restrict__ ngroups,
                                                               const uint32_t* __restrict__ P,
                                                               const uint32_t* __restrict__ tile_lo,
                                                               const hn_vrec* __restrict__ rec,
                                                               const int32_t* __restrict__ arena, int step,
                                                               uint32_t* __restrict__ weight) {
    __shared__ TcLb sh;
    const uint32_t total = *ngroups;
    const int64_t ntiles = ((int64_t)total + TC_TILE - 1) / TC_TILE;
    for (int64_t t = (int64_t)blockIdx.x * step; t < ntiles; t += (int64_t)gridDim.x * step) {
        uint32_t unit[TC_IPT];
        const TcLoc c = tc_locate(P, nv, total, tile_lo, t, ntiles, sh,
                                  [&](int64_t s) { return (uint32_t)(rec[s].off / UNIT_SLOTS); }, unit);
#pragma unroll
        for (int j = 0; j < TC_IPT; j++) {
            const int64_t at = (int64_t)unit[j] * UNIT_SLOTS + (int64_t)c.k[j] * TC_G;
            const int64_t n = c.seg[j] < 0 ? 0 : (int64_t)rec[c.seg[j]].deg - (int64_t)c.k[j] * TC_G;
            for (int e = 0; e < TC_G; e++) {
                const bool in = e < n;
                const uint64_t some = __ballot(in);
                if (some == 0) break;
                const int first = __ffsll((unsigned long long)some) - 1;
                const int32_t v = in ? arena[at + e] : -1, lead = __shfl(v, first, WAVE);
                const uint32_t same = (uint32_t)__popcll(__ballot(v == lead));
                if (in && (v != lead || (int)__lane_id() == first)) atomicAdd(weight + v, v == lead ? same : 1u);
            }
        }
        __syncthreads();
    }
}

// Stored rows -> lists (ORIENT: only the entries up the degree order).  A lane
// holds eight entries of one row; the lanes of a wave that hold the same row
// claim its next places, in both of its rows, with one atomic, or none if they hold
// all of it (four million rows of four entries: 461 us with one for each, 440 so;
// of one entry: 457, 274).
// Stored rows need the codes of hubs only, and the L2 holds a bit per vertex that says which
// are (four million rows of four entries 442 us with a look-up for every entry, 272 so;
// 16 M rows 1,880 and 1,230); degree orders need every entry's degree.
typedef int32_t TcVec __attribute__((ext_vector_type(4)));
template <bool ORIENT>
__global__ __launch_bounds__(BLOCK) void tc_rows_kernel(int64_t nv, const uint32_t* __restrict__ ngroups,
                                                        const uint32_t* __restrict__ P,
                                                        const uint32_t* __restrict__ tile_lo,
                                                        const hn_vrec* __restrict__ rec,
                                                        const int32_t* __restrict__ arena,
                                                        const uint2* __restrict__ wc,
                                                        const uint64_t* __restrict__ hubs, TcRow* __restrict__ row,
                                                        uint16_t* __restrict__ codes, uint32_t* __restrict__ ids,
                                                        TcCtl* __restrict__ ctl) {
    __shared__ TcLb sh;
    const uint32_t total = *ngroups;
    const int64_t ntiles = ((int64_t)total + TC_TILE - 1) / TC_TILE;
    const int lane = __lane_id();
    bool twice = false;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint32_t unit[TC_IPT];
        const TcLoc c = tc_locate(P, nv, total, tile_lo, t, ntiles, sh,
                                  [&](int64_t s) { return (uint32_t)(rec[s].off / UNIT_SLOTS); }, unit);
        int32_t a[TC_IPT][TC_G], prev[TC_IPT], deg[TC_IPT];
#pragma unroll
        for (int j = 0; j < TC_IPT; j++) {
            const int64_t at = (int64_t)unit[j] * UNIT_SLOTS + (int64_t)c.k[j] * TC_G;
            const TcVec p = *reinterpret_cast<const TcVec*>(arena + at), q = *reinterpret_cast<const TcVec*>(arena + at + 4);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                a[j][e] = p[e];
                a[j][4 + e] = q[e];
            }
            prev[j] = c.k[j] ? arena[at - 1] : -1;
            deg[j] = rec[c.seg[j] >= 0 ? c.seg[j] : 0].deg;
        }
#pragma unroll
        for (int j = 0; j < TC_IPT; j++) {
            const int64_t n = c.seg[j] >= 0 ? (int64_t)deg[j] - (int64_t)c.k[j] * TC_G : 0;
            const int32_t u = (int32_t)c.seg[j];
            uint2 x[TC_G];
#pragma unroll
            for (int e = 0; e < TC_G; e++) {
                if constexpr (ORIENT) {
                    x[e] = wc[e < n ? a[j][e] : 0];
                } else {
                    const uint32_t v = e < n ? (uint32_t)a[j][e] : 0u;
                    x[e].x = !hubs || (hubs[v / WAVE] >> (v % WAVE) & 1u) ? 1u : 0u;   // (no bits: all are)
                }
            }
            if constexpr (!ORIENT)
#pragma unroll
                for (int e = 0; e < TC_G; e++) x[e].y = !hubs ? (uint32_t)a[j][e] : x[e].x ? wc[e < n ? a[j][e] : 0].y : TC_ID;
            uint32_t keep = 0, hubs = 0;
#pragma unroll
            for (int e = 0; e < TC_G; e++) {
                const int32_t v = a[j][e];
                const bool k = e < n && (!ORIENT || (uint32_t)deg[j] < x[e].x || ((uint32_t)deg[j] == x[e].x && u < v));
                keep |= (uint32_t)k << e;
                hubs |= (uint32_t)(k && !(x[e].y & TC_ID)) << e;
                twice = twice || (e < n && v == (e ? a[j][e - 1] : prev[j]));
            }
            // both counts in one word: a wave holds at most 512 entries
            const uint32_t cnt = (uint32_t)__popc(hubs) | (uint32_t)__popc(keep & ~hubs) << 16;
            const uint32_t inc = wave_inclusive_scan(cnt);
            const int32_t up = __shfl_up(u, 1, WAVE);
            const uint64_t heads = __ballot(lane == 0 || u != up);
            const int head = 63 - __clzll((long long)(heads & (lanemask_lt() | (1ull << lane))));
            const uint64_t above = lane == WAVE - 1 ? 0ull : heads & (~0ull << (lane + 1));
            const int tail = above ? __ffsll((unsigned long long)above) - 2 : WAVE - 1;
            const uint32_t before = __shfl(inc - cnt, head, WAVE);
            const uint32_t sum = __shfl(inc, tail, WAVE) - before;
            unsigned long long at = 0;
            if (lane == head && sum) {
                unsigned long long* cur = reinterpret_cast<unsigned long long*>(&row[u].n16);
                const unsigned long long n2 = (unsigned long long)(sum & 0xFFFFu) | (unsigned long long)(sum >> 16) << 32;
                if (c.k[j] == 0 && (tail - head + 1) * TC_G >= deg[j]) *cur = n2;
                else at = atomicAdd(cur, n2);
            }
            const uint32_t at16 = __shfl((uint32_t)at, head, WAVE), at32 = __shfl((uint32_t)(at >> 32), head, WAVE);
            if (keep) {
                const uint32_t mine = inc - cnt - before;
                const int64_t base = (t * TC_TILE + (int64_t)j * BLOCK + threadIdx.x - c.k[j]) * TC_G;   // (as row[u].base)
                uint16_t* o16 = codes + base + at16 + (mine & 0xFFFFu);
                uint32_t* o32 = ids + base + at32 + (mine >> 16);
#pragma unroll
                for (int e = 0; e < TC_G; e++) {
                    if ((hubs >> e) & 1u) *o16++ = (uint16_t)x[e].y;
                    else if ((keep >> e) & 1u) *o32++ = (uint32_t)a[j][e];
                }
            }
        }
        __syncthreads();
    }
    if (__ballot(twice) && lane == 0) ctl->repeats = 1u;   // every writer stores the same value
}

// The lists' padding, and two bits per vertex: its list is long enough for it to be an
// owner (whose counter of grouped edges starts at 0), or one that tc_small_kernel takes.
// Vertices without entries, all but a few of some graphs, cost this pass and the
// later ones their bits only (16 M vertices with a thousand edges, where it was
// their 16-byte rows and counters: 72 -> 28 us here, 52 -> 22 there, 129 -> 58 in the
// scans; stored 663 -> 535 in all, oriented 646 -> 540).
constexpr int TC_PAD_WORDS = 4;   // of 64 vertices to a wave
__global__ __launch_bounds__(BLOCK) void tc_pad_kernel(int64_t nv, const uint64_t* __restrict__ some,
                                                       const TcRow* __restrict__ row, uint16_t* __restrict__ codes,
                                                       uint32_t* __restrict__ ids, uint32_t most,
                                                       uint64_t* __restrict__ owner, uint64_t* __restrict__ small,
                                                       uint32_t* __restrict__ gcnt) {
    const int64_t w0 = ((int64_t)blockIdx.x * NWAVES + threadIdx.x / WAVE) * TC_PAD_WORDS, words = (nv + WAVE - 1) / WAVE;
    const int lane = __lane_id();
    TcRow r[TC_PAD_WORDS];
#pragma unroll
    for (int j = 0; j < TC_PAD_WORDS; j++) {
        const bool any = w0 + j < words && (some[w0 + j] >> lane & 1u);
        r[j] = any ? row[(w0 + j) * WAVE + lane] : TcRow{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < TC_PAD_WORDS; j++) {
        const uint64_t big = __ballot(r[j].len() > most), few = __ballot(r[j].len() >= 2 && r[j].len() <= most);
        if (lane == 0 && w0 + j < words) {
            owner[w0 + j] = big;
            small[w0 + j] = few;
        }
        if (r[j].len() > most) gcnt[(w0 + j) * WAVE + lane] = 0;
        for (uint32_t i = r[j].n16; i & (TC_G - 1); i++) codes[(int64_t)r[j].base * TC_G + i] = (uint16_t)TC_PAD16;
        for (uint32_t i = r[j].n32; i & (TC_G - 1); i++) ids[(int64_t)r[j].base * TC_G + i] = TC_PAD;
    }
}

// entry i of a list, as a vertex
__device__ __forceinline__ uint32_t tc_entry(const TcRow& r, uint32_t i, const uint16_t* __restrict__ codes,
                                             const uint32_t* __restrict__ ids, const uint32_t* __restrict__ hub) {
    return i < r.n16 ? hub[codes[(int64_t)r.base * TC_G + i]] : ids[(int64_t)r.base * TC_G + (i - r.n16)];
}

// ---- edges whose longer list is the destination's, grouped by it (where an
// owner's edges cannot be read from its stored row), over the same partition
// FILL = false: the edge's place in its group (TC_PAD: not grouped); FILL = true: the sources at their places
// A hub's group is counted in TC_LANES parts (by workgroup, the same in both passes),
// as atomics on one counter take 10 ns each: R-MAT s18 oriented, 319 us in one part, 118 so.
// Otherwise bound by the lookups of the entries' lists: only owners' are looked up, by a
// bit that the L2 holds (four million vertices of four entries: 525 us without, 217 so).
// 512 entries without a grouped edge (a wave's) have that noted (`placed`) and no places, and
// a tile without any is not read again (the same vertices, of which few are owners: 213
// and 119 us, 122 and 5 so; by eight entries, places would be parts of lines, and 256 K
// vertices of 64 entries take 35 us more to read them).
template <bool FILL>
__global__ __launch_bounds__(BLOCK) void tc_group_kernel(int64_t nv, const uint32_t* __restrict__ ngroups,
                                                         const uint32_t* __restrict__ P,
                                                         const uint32_t* __restrict__ tile_lo, int sym,
                                                         const TcCtl* __restrict__ ctl, const TcRow* __restrict__ row,
                                                         const uint64_t* __restrict__ owner,
                                                         const uint16_t* __restrict__ codes,
                                                         const uint32_t* __restrict__ ids,
                                                         const uint32_t* __restrict__ hub, uint32_t* __restrict__ gcnt,
                                                         uint32_t* __restrict__ part, int64_t nhub,
                                                         uint32_t* __restrict__ place, uint8_t* __restrict__ placed,
                                                         const uint32_t* __restrict__ goff, uint32_t* __restrict__ members) {
    if (sym && !ctl->repeats) return;
    uint32_t* const mine = part + (blockIdx.x % TC_LANES) * nhub;
    __shared__ TcLb sh;
    const uint32_t total = *ngroups;
    const int64_t ntiles = ((int64_t)total + TC_TILE - 1) / TC_TILE;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint8_t* const some = placed + t * (TC_TILE / WAVE);   // of a wave's 64 groups
        bool fill[TC_IPT] = {};
        if constexpr (FILL) {
#pragma unroll
            for (int j = 0; j < TC_IPT; j++) fill[j] = some[j * NWAVES + threadIdx.x / WAVE] != 0;
            static_assert(TC_TILE / WAVE == 8, "one word has all");
            if (*reinterpret_cast<const uint64_t*>(some) == 0) continue;
        }
        uint32_t unused[TC_IPT];
        const TcLoc c = tc_locate(P, nv, total, tile_lo, t, ntiles, sh, [&](int64_t) { return 0u; }, unused);
#pragma unroll
        for (int j = 0; j < TC_IPT; j++) {
            // entries [8k, 8k + 8) of a list, which may end before its stored row
            bool in = (FILL ? fill[j] : true) && c.seg[j] >= 0;
            const uint32_t u = in ? (uint32_t)c.seg[j] : 0u, i0 = c.k[j] * TC_G;
            const TcRow r = in ? row[u] : TcRow{0u, 0u, 0u, 0u};
            const uint32_t lu = r.len();
            const int64_t at = (int64_t)r.base * TC_G;
            in = in && lu >= 2 && i0 < lu;
            uint32_t q[TC_G], v[TC_G], lv[TC_G];
            if (in) {
#pragma unroll
                for (int e = 0; e < TC_G; e++) {
                    const uint32_t i = i0 + e;
                    q[e] = i < r.n16 ? codes[at + i] : TC_PAD;
                    v[e] = i >= r.n16 && i < lu ? ids[at + (i - r.n16)] : u;
                }
#pragma unroll
                for (int e = 0; e < TC_G; e++)
                    if (q[e] != TC_PAD) v[e] = hub[q[e]];
            }
            if constexpr (FILL) {
                if (!in) continue;
#pragma unroll
                for (int e = 0; e < TC_G; e++) {
                    const uint32_t pl = i0 + e < lu ? place[at + i0 + e] : TC_PAD;
                    if (pl != TC_PAD) members[(int64_t)goff[v[e]] + (q[e] != TC_PAD ? mine[q[e]] : 0u) + pl] = u;
                }
            } else {
                bool any = false;
                if (in) {
                    uint64_t big[TC_G];
#pragma unroll
                    for (int e = 0; e < TC_G; e++) big[e] = owner[v[e] / WAVE];
#pragma unroll
                    for (int e = 0; e < TC_G; e++) lv[e] = v[e] != u && (big[e] >> (v[e] % WAVE) & 1u) ? row[v[e]].len() : 0u;
#pragma unroll
                    for (int e = 0; e < TC_G; e++) any = any || (i0 + e < lu && lv[e] > lu);
                }
                const bool write = __ballot(any) != 0;
                if (write && in)
#pragma unroll
                    for (int e = 0; e < TC_G; e++)
                        if (i0 + e < lu)
                            place[at + i0 + e] = lv[e] > lu ? atomicAdd(q[e] != TC_PAD ? mine + q[e] : gcnt + v[e], 1u) : TC_PAD;
                if (__lane_id() == 0) some[j * NWAVES + threadIdx.x / WAVE] = write ? 1 : 0;
            }
        }
        __syncthreads();
    }
}

// a hub's parts: their starts within its group, and the group's size
__global__ __launch_bounds__(BLOCK) void tc_parts_kernel(int sym, const TcCtl* __restrict__ ctl, int64_t nhub,
                                                         const uint32_t* __restrict__ hub, uint32_t* __restrict__ part,
                                                         uint32_t* __restrict__ gcnt) {
    if (sym && !ctl->repeats) return;
    const int64_t q = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (q >= nhub || q >= (int64_t)ctl->hubs) return;
    uint32_t at = 0;
    for (int p = 0; p < TC_LANES; p++) {
        const uint32_t c = part[p * nhub + q];
        part[p * nhub + q] = at;
        at += c;
    }
    gcnt[hub[q]] = at;
}

// ---- owners: where their grouped edges start, and tasks of up to TC_CAND candidates
// (low and high half of one scan, which looks at owners only)
struct OwnerIn {
    const uint64_t* owner;
    const TcRow* row;
    const uint32_t* gcnt;
    const hn_vrec* rec;
    const TcCtl* ctl;
    int sym;
    __device__ __forceinline__ uint64_t operator()(int64_t v) const {
        if (!(owner[v / WAVE] >> (v % WAVE) & 1u)) return 0u;
        const uint32_t n = gcnt[v];
        const uint32_t cand = sym && !ctl->repeats ? (uint32_t)rec[v].deg : row[v].len() + n;
        return (uint64_t)n | (uint64_t)((cand + TC_CAND - 1) / TC_CAND) << 32;
    }
};
struct OwnerOut {
    uint32_t* goff;
    uint2* task;
    __device__ __forceinline__ void operator()(int64_t v, uint64_t ex, uint64_t x) const {
        if (x) goff[v] = (uint32_t)ex;
        const uint32_t first = (uint32_t)(ex >> 32);
        tc_spread((uint32_t)v, first, first + (uint32_t)(x >> 32), [&](uint32_t w, uint32_t a, uint32_t k) { task[k] = make_uint2(w, k - a); });
    }
};

struct OwnerShared {
    uint32_t bits[(TC_HUBS + 1) / 32];
    uint32_t hash[TC_HASH];
    uint32_t y[TC_STEP], base[TC_STEP], n16[TC_STEP], n32[TC_STEP];   // the edges listed: vertex and rows of the shorter list
    uint32_t cls[TC_ORDER];
    uint32_t tail;
    uint2 task;
    uint32_t cur, end, tried;        // the first lane's tickets (in LDS: it has no registers to spare)
};
static_assert(sizeof(OwnerShared) * 8 <= 160 * 1024, "eight workgroups fill a CU's LDS");

// Two sizes of table: beside the hubs' bits, or, where these are done with, in their place.
template <uint32_t SLOTS>
__device__ __forceinline__ uint32_t tc_slot(uint32_t id) { return (id * 2654435761u) >> (__builtin_clz(SLOTS) + 1); }
template <uint32_t SLOTS>
__device__ __forceinline__ void tc_fill(uint32_t* table, const uint32_t* __restrict__ ids, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < SLOTS; i += BLOCK) table[i] = TC_PAD;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += BLOCK) {
        const uint32_t q = ids[i];
        for (uint32_t s = tc_slot<SLOTS>(q);; s = (s + 1) & (SLOTS - 1)) {
            const uint32_t z = atomicCAS(table + s, TC_PAD, q);
            if (z == TC_PAD || z == q) break;
        }
    }
}
template <uint32_t SLOTS>
__device__ __forceinline__ bool tc_holds(const uint32_t* table, uint32_t q) {
    for (uint32_t s = tc_slot<SLOTS>(q);; s = (s + 1) & (SLOTS - 1)) {
        const uint32_t z = table[s];
        if (z == q || z == TC_PAD) return z == q;
    }
}

__device__ __forceinline__ uint32_t tc_test(const OwnerShared& sh, const uint4& x) {
    const uint32_t q[4] = {x.x, x.y, x.z, x.w};
    uint32_t k = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {   // two codes a word: bit (code & 31) of word code >> 5
        const uint32_t lo = q[e], hi = q[e] >> 16;
        k += (sh.bits[(lo >> 5) & 2047u] >> (lo & 31)) & 1u;
        k += (sh.bits[hi >> 5] >> (hi & 31)) & 1u;
    }
    return k;
}

// The listed edges' shorter lists against the owner's set: a team of eight
// lanes per list, eight codes per lane and group.  The lists are sorted by
// length class, so that the teams of a wave stay together: TC_DEPTH groups of one
// list in flight while lists are longer than a team's step, then TC_DEPTH lists.
enum TcTail { TC_NONE, TC_HASHED, TC_SORTED };
struct TcSorted {   // an owner's stored row
    const int32_t* entry;
    int32_t deg;
    const uint2* wc;    // where only the entries up the degree order are in its list, else null
    uint32_t owner;
    __device__ __forceinline__ bool has(uint32_t q) const {
        int32_t lo = 0, hi = deg;
        while (lo < hi) {
            const int32_t mid = (lo + hi) >> 1;
            if ((uint32_t)entry[mid] < q) lo = mid + 1; else hi = mid;
        }
        if (lo == deg || (uint32_t)entry[lo] != q) return false;
        if (!wc) return true;
        const uint32_t w = wc[q].x;
        return (uint32_t)deg < w || ((uint32_t)deg == w && owner < q);
    }
};
template <TcTail TAIL>
__device__ __forceinline__ uint32_t tc_ids(const OwnerShared& sh, uint32_t it, int sub, const uint32_t* __restrict__ ids,
                                           const TcSorted& sorted) {
    uint32_t c = 0;
    if constexpr (TAIL != TC_NONE) {
        const uint32_t* li = ids + (int64_t)sh.base[it] * TC_G;
        const uint32_t n32 = sh.n32[it];
        for (uint32_t i = sub; i < n32; i += TC_TEAM) {
            const uint32_t q = li[i];
            if constexpr (TAIL == TC_HASHED) c += tc_holds<TC_HASH>(sh.hash, q) ? 1u : 0u;
            if constexpr (TAIL == TC_SORTED) c += sorted.has(q) ? 1u : 0u;
        }
    }
    return c;
}
// the sums of eight lanes in lanes 7 and 15 of every row
__device__ __forceinline__ uint32_t tc_team_sum(uint32_t c) {
    c += dpp_move<0x111, 0xf>(c);
    c += dpp_move<0x112, 0xf>(c);
    c += dpp_move<0x114, 0xf>(c);
    return c;
}
template <TcTail TAIL>
__device__ __forceinline__ void tc_walk(const OwnerShared& sh, uint32_t nlong, uint32_t n,
                                        const uint16_t* __restrict__ codes, const uint32_t* __restrict__ ids,
                                        const TcSorted& sorted,
                                        unsigned long long* __restrict__ per_vertex, uint64_t& acc) {
    constexpr uint32_t TEAMS = BLOCK / TC_TEAM;
    const int sub = threadIdx.x & (TC_TEAM - 1);
    const uint4* rows = reinterpret_cast<const uint4*>(codes);
    uint32_t it = threadIdx.x / TC_TEAM;
    for (; it < nlong; it += TEAMS) {
        const uint4* list = rows + sh.base[it];
        const uint32_t ng = (sh.n16[it] + TC_G - 1) / TC_G;
        uint32_t c = tc_ids<TAIL>(sh, it, sub, ids, sorted);
        for (uint32_t g0 = sub; g0 < ng; g0 += TC_TEAM * TC_DEPTH) {
            uint4 x[TC_DEPTH];
#pragma unroll
            for (int d = 0; d < TC_DEPTH; d++) {
                const uint32_t g = g0 + d * TC_TEAM;
                if (__ballot(g < ng) == 0) break;
                x[d] = list[g < ng ? g : g0];
            }
#pragma unroll
            for (int d = 0; d < TC_DEPTH; d++) {
                const bool in = g0 + d * TC_TEAM < ng;
                if (__ballot(in) == 0) break;
                const uint32_t k = tc_test(sh, x[d]);
                c += in ? k : 0u;
            }
        }
        acc += c;
        c = tc_team_sum(c);
        if (sub == TC_TEAM - 1 && c && per_vertex) atomicAdd(per_vertex + sh.y[it], (unsigned long long)c);
    }
    for (; it < n; it += TEAMS * TC_DEPTH) {
        uint4 x[TC_DEPTH];
        bool in[TC_DEPTH];
#pragma unroll
        for (int d = 0; d < TC_DEPTH; d++) {
            const uint32_t i = min(it + d * TEAMS, n - 1);
            in[d] = it + d * TEAMS < n && (uint32_t)sub * TC_G < sh.n16[i];
            x[d] = rows[(int64_t)sh.base[i] + (in[d] ? sub : 0)];
        }
#pragma unroll
        for (int d = 0; d < TC_DEPTH; d++) {
            const uint32_t i = it + d * TEAMS;
            if (i >= n) break;
            const uint32_t k = tc_test(sh, x[d]);
            uint32_t c = (in[d] ? k : 0u) + tc_ids<TAIL>(sh, i, sub, ids, sorted);
            acc += c;
            c = tc_team_sum(c);
            if (sub == TC_TEAM - 1 && c && per_vertex) atomicAdd(per_vertex + sh.y[i], (unsigned long long)c);
        }
    }
}

// The same against a table in the bits' place: ids only.  An owner with that many has
// neighbours with lists like its own, so a lane has eight ids on their way (14 cliques of
// 5,000: 1.60 s with one, 0.89 so; in tc_walk they would cost registers that the walks of
// codes need: R-MAT s22 2 % slower).
__device__ __forceinline__ void tc_walk_wide(const OwnerShared& sh, uint32_t n, const uint32_t* __restrict__ ids,
                                             unsigned long long* __restrict__ per_vertex, uint64_t& acc) {
    constexpr uint32_t STEP = TC_TEAM * 4, DEPTH = 2;
    const uint32_t sub = threadIdx.x & (TC_TEAM - 1);
    for (uint32_t it = threadIdx.x / TC_TEAM; it < n; it += BLOCK / TC_TEAM) {
        const uint32_t* li = ids + (int64_t)sh.base[it] * TC_G;
        const uint32_t n32 = sh.n32[it];
        uint32_t c = 0, i0 = 0;
        auto test = [&](uint32_t q) { c += tc_holds<TC_WIDE_HASH>(sh.bits, q) ? 1u : 0u; };
        for (; i0 + STEP * DEPTH <= n32; i0 += STEP * DEPTH) {
            uint4 x[DEPTH];
#pragma unroll
            for (int d = 0; d < (int)DEPTH; d++) x[d] = *reinterpret_cast<const uint4*>(li + i0 + d * STEP + sub * 4);
#pragma unroll
            for (int d = 0; d < (int)DEPTH; d++) {
                test(x[d].x);
                test(x[d].y);
                test(x[d].z);
                test(x[d].w);
            }
        }
        for (uint32_t i = i0 + sub; i < n32; i += TC_TEAM) test(li[i]);
        acc += c;
        c = tc_team_sum(c);
        if (sub == TC_TEAM - 1 && c && per_vertex) atomicAdd(per_vertex + sh.y[it], (unsigned long long)c);
    }
}

// Bound by the sectors of the shorter lists that miss the L2: on R-MAT s22 360 M of
// the 400 M that the walks touch, 7.4 ms at the 48 G/s that scattered sector reads
// reach here; LDS and vector units are a third busy.
__global__ __launch_bounds__(BLOCK) void tc_owner_kernel(int orient, int sym, const hn_vrec* __restrict__ rec,
                                                         const int32_t* __restrict__ arena,
                                                         const uint2* __restrict__ wc, const uint2* __restrict__ task,
                                                         const TcRow* __restrict__ row,
                                                         const uint16_t* __restrict__ codes,
                                                         const uint32_t* __restrict__ ids,
                                                         const uint32_t* __restrict__ hub,
                                                         const uint32_t* __restrict__ gcnt,
                                                         const uint32_t* __restrict__ goff,
                                                         const uint32_t* __restrict__ members, TcCtl* __restrict__ ctl,
                                                         unsigned long long* __restrict__ per_vertex) {
    __shared__ OwnerShared sh;
    const uint32_t ntask = (uint32_t)(ctl->owned >> 32);
    const bool repeats = ctl->repeats != 0;
    const bool stored = sym && !repeats;
    uint64_t acc = 0;
    for (int i = threadIdx.x; i < (int)(TC_HUBS + 1) / 32; i += BLOCK) sh.bits[i] = 0;
    // The next task is taken while this one runs.  Tickets are for `chunk` tasks, of
    // one of TC_LANES interleaved shares; the others' once that one is used up.  (One
    // ticket for each of R-MAT s22's 640 K tasks, from one counter, was what
    // bounded the kernel: 10.1 ms, 7.6 ms so.)
    const uint32_t chunk = min(max(ntask / (gridDim.x * 32u), 1u), 8u);
    if (threadIdx.x == 0) sh.cur = sh.end = sh.tried = 0;
    auto next = [&]() {
        while (sh.cur >= sh.end) {
            if (sh.tried == TC_LANES) return make_uint2(0u, TC_PAD);
            const uint32_t share = (blockIdx.x + sh.tried) % TC_LANES;
            uint32_t* at = &ctl->ticket[share].v;
            const uint32_t seen = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t first = ((uint64_t)seen * TC_LANES + share) * chunk;
            uint64_t lo = first;
            if (first < ntask) lo = ((uint64_t)atomicAdd(at, 1u) * TC_LANES + share) * chunk;
            if (lo >= ntask) {
                sh.tried++;
                continue;
            }
            sh.cur = (uint32_t)lo;
            sh.end = (uint32_t)min(lo + chunk, (uint64_t)ntask);
        }
        return task[sh.cur++];
    };
    uint2 ahead = make_uint2(0u, TC_PAD);
    if (threadIdx.x == 0) sh.task = next();
    __syncthreads();
    for (;;) {
        const uint2 tk = sh.task;
        if (tk.y == TC_PAD) break;
        if (threadIdx.x == 0) ahead = next();
        const uint32_t x = tk.x;
        const TcRow rx = row[x];
        const hn_vrec sx = rec[x];
        const uint32_t lx = rx.len(), cand = stored ? (uint32_t)sx.deg : lx + gcnt[x];
        const uint32_t c0 = tk.y * TC_CAND, c1 = min(c0 + TC_CAND, cand);
        const int64_t at = (int64_t)rx.base * TC_G;
        // An entry that is stored twice must not lie in two tables, or it counts twice:
        // with repeats, what does not fit one table is searched.
        const bool search = repeats ? rx.n32 > (rx.n16 ? TC_TAIL : TC_WIDE_TAIL) : !orient && rx.n32 > TC_SEARCH;
        const TcSorted sorted = {arena + sx.off, sx.deg, orient ? wc : nullptr, x};
        // the set: the hubs' bits and the first ids, then the other ids in tables that
        // take the bits' place (alone where no hub is listed)
        const bool narrow = rx.n16 || search || rx.n32 <= TC_TAIL;
        const uint32_t near = narrow ? min(rx.n32, TC_TAIL) : 0u;
        const uint32_t passes = search ? 1u : (narrow ? 1u : 0u) + (rx.n32 - near + TC_WIDE_TAIL - 1) / TC_WIDE_TAIL;
        for (uint32_t p = 0; p < passes; p++) {
            const bool wide = !narrow || p > 0;
            if (wide) {
                const uint32_t from = near + (narrow ? p - 1 : p) * TC_WIDE_TAIL;
                tc_fill<TC_WIDE_HASH>(sh.bits, ids + at + from, min(rx.n32 - from, TC_WIDE_TAIL));
            } else {
                for (uint32_t i = threadIdx.x; i < rx.n16; i += BLOCK) {
                    const uint32_t q = codes[at + i];
                    atomicOr(&sh.bits[q >> 5], 1u << (q & 31));
                }
                if (near && !search) tc_fill<TC_HASH>(sh.hash, ids + at, near);
            }
            for (uint32_t b = c0; b < c1; b += TC_STEP) {
                if (threadIdx.x < TC_ORDER) sh.cls[threadIdx.x] = 0;
                __syncthreads();   // (the set too)
                uint32_t y[TC_STEP / BLOCK], cl[TC_STEP / BLOCK], pos[TC_STEP / BLOCK];
                TcRow ry[TC_STEP / BLOCK];
#pragma unroll
                for (int j = 0; j < TC_STEP / BLOCK; j++) {
                    const uint32_t i = b + j * BLOCK + threadIdx.x;
                    y[j] = x;
                    if (i < c1)
                        y[j] = stored ? (uint32_t)arena[sx.off + i]
                                      : i < lx ? tc_entry(rx, i, codes, ids, hub) : members[(int64_t)goff[x] + (i - lx)];
                    ry[j] = row[y[j]];
                }
#pragma unroll
                for (int j = 0; j < TC_STEP / BLOCK; j++) {
                    const uint32_t ly = ry[j].len();
                    // shorter lists, and lists as long of edges whose source x is
                    bool take = y[j] != x && ly != 0 && ly <= lx;
                    if (stored && take && ly == lx) {
                        const uint32_t wx = wc[x].x, wy = wc[y[j]].x;
                        take = wx < wy || (wx == wy && x < y[j]);
                    }
                    // classes by steps of a team, the longest first
                    const uint32_t steps = (ry[j].n16 + TC_TEAM * TC_G - 1) / (TC_TEAM * TC_G);
                    cl[j] = take ? TC_ORDER - 1 - min(steps, (uint32_t)TC_ORDER - 1) : TC_PAD;
                    pos[j] = take ? atomicAdd(&sh.cls[cl[j]], 1u) : 0u;
                }
                __syncthreads();
                uint32_t n = 0;
                if (threadIdx.x < WAVE) {
                    const uint32_t k = threadIdx.x < TC_ORDER ? sh.cls[threadIdx.x] : 0u;
                    const uint32_t inc = wave_inclusive_scan(k);
                    if (threadIdx.x < TC_ORDER) sh.cls[threadIdx.x] = inc - k;
                    if (threadIdx.x == WAVE - 1) sh.tail = inc;
                }
                __syncthreads();
                n = sh.tail;
                const uint32_t nlong = sh.cls[TC_ORDER - 2];   // of the last two classes are one step or none
#pragma unroll
                for (int j = 0; j < TC_STEP / BLOCK; j++)
                    if (cl[j] != TC_PAD) {
                        const uint32_t k = sh.cls[cl[j]] + pos[j];
                        sh.y[k] = y[j];
                        sh.base[k] = ry[j].base;
                        sh.n16[k] = ry[j].n16;
                        sh.n32[k] = ry[j].n32;
                    }
                __syncthreads();
                if (rx.n32 == 0) tc_walk<TC_NONE>(sh, nlong, n, codes, ids, sorted, per_vertex, acc);
                else if (search) tc_walk<TC_SORTED>(sh, nlong, n, codes, ids, sorted, per_vertex, acc);
                else if (wide) tc_walk_wide(sh, n, ids, per_vertex, acc);
                else tc_walk<TC_HASHED>(sh, nlong, n, codes, ids, sorted, per_vertex, acc);
                __syncthreads();
            }
        }
        if (passes > 1 || !narrow)
            for (uint32_t i = threadIdx.x; i < TC_WIDE_HASH; i += BLOCK) sh.bits[i] = 0;
        else
            for (uint32_t i = threadIdx.x; i < rx.n16; i += BLOCK) sh.bits[codes[at + i] >> 5] = 0;
        if (threadIdx.x == 0) sh.task = ahead;
        __syncthreads();
    }
    acc = wave_reduce_sum(acc);
    if (__lane_id() == 0 && acc) atomicAdd(&ctl->total[(blockIdx.x + threadIdx.x / WAVE) % TC_SUMS].v, (unsigned long long)acc);
}

// The entries of list s that list l holds too, group by group; what pads l equals
// no entry, and s is masked.
__device__ __forceinline__ uint32_t tc_common(const TcRow& s, const TcRow& l, const uint16_t* __restrict__ codes,
                                              const uint32_t* __restrict__ ids) {
    uint32_t c = 0;
    const uint4* c4 = reinterpret_cast<const uint4*>(codes);
    for (uint32_t gs = 0; gs * TC_G < s.n16; gs++) {
        const uint4 a = c4[(int64_t)s.base + gs];
        const uint32_t x[4] = {a.x, a.y, a.z, a.w};
        uint32_t m = 0;
        for (uint32_t gl = 0; gl * TC_G < l.n16; gl++) {
            const uint4 b = c4[(int64_t)l.base + gl];
            const uint32_t y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < TC_G; e++) {
                const uint32_t q = x[e / 2] >> (16 * (e & 1)) & 0xFFFFu;
                bool in = false;
#pragma unroll
                for (int f = 0; f < 4; f++) in = in || q == (y[f] & 0xFFFFu) || q == y[f] >> 16;
                m |= (uint32_t)in << e;
            }
        }
        c += (uint32_t)__popc(m & ((1u << min(s.n16 - gs * TC_G, (uint32_t)TC_G)) - 1u));
    }
    const uint4* i4 = reinterpret_cast<const uint4*>(ids);
    for (uint32_t gs = 0; gs * 4 < s.n32; gs++) {
        const uint4 a = i4[(int64_t)s.base * 2 + gs];
        const uint32_t x[4] = {a.x, a.y, a.z, a.w};
        uint32_t m = 0;
        for (uint32_t gl = 0; gl * 4 < l.n32; gl++) {
            const uint4 b = i4[(int64_t)l.base * 2 + gl];
#pragma unroll
            for (int e = 0; e < 4; e++) m |= (uint32_t)(x[e] == b.x || x[e] == b.y || x[e] == b.z || x[e] == b.w) << e;
        }
        c += (uint32_t)__popc(m & ((1u << min(s.n32 - gs * 4, 4u)) - 1u));
    }
    return c;
}

// Edges between two lists of at most `most` entries: a lane per edge, TC_SMALL
// lanes per source, twice where it has more.  The chain source row, entry, hub, row, list is what bounds
// it, so a lane starts four of them at once; a thread per source, one entry after
// the other, took 330 us on a graph of a thousand vertices.
// An owner's task is a longer chain, 20 us for a handful of candidates, and its edges are
// grouped first: 260 K vertices with 16 entries to others took 1.65 ms where lists of
// 17 to 32 entries were owners', 0.60 so; 100 K, 718 and 307 us.  Not where few waves
// share the work (R-MAT s12 oriented, 140 us, 182 so; s17 690 and 715), nor on symmetric
// storage, where nothing is grouped (R-MAT s22 9.4 and 10.4 ms).
// A wave's sources are those of `per` vertices, its lanes' own rows: 16, one step at
// most, or 64 where there are waves enough all the same (16 M vertices with
// a thousand edges: 186 us with every lane reading its source's row, 51 so; four million of
// four entries: 975, 690; R-MAT s12 is 20 % slower with 64, 16 M vertices are so with 16).
constexpr int TC_SRC = 4;
constexpr int64_t TC_WIDE = 1 << 20;
__global__ __launch_bounds__(BLOCK) void tc_small_kernel(int64_t nv, int per, uint32_t most, const uint64_t* __restrict__ small,
                                                         const TcRow* __restrict__ row,
                                                         const uint16_t* __restrict__ codes,
                                                         const uint32_t* __restrict__ ids,
                                                         const uint32_t* __restrict__ hub, TcCtl* __restrict__ ctl,
                                                         unsigned long long* __restrict__ per_vertex) {
    const int lane = __lane_id(), team = lane / TC_SMALL;
    const uint32_t sub = lane % TC_SMALL;
    const int64_t w0 = ((int64_t)blockIdx.x * NWAVES + threadIdx.x / WAVE) * per;
    if (w0 >= nv) return;
    const bool has = lane < per && (small[w0 / WAVE] >> (w0 % WAVE) >> lane & 1u);   // (no bits from nv on)
    const uint64_t m = __ballot(has);
    if (m == 0) return;
    const TcRow own = has ? row[w0 + lane] : TcRow{0u, 0u, 0u, 0u};
    uint64_t acc = 0;
    // entries [i0, i0 + TC_SMALL) of the lists that have them
    for (uint32_t i0 = 0; i0 < most; i0 += TC_SMALL) {
        const bool src = own.len() > i0;
        const uint64_t ms = __ballot(src);
        const int nsrc = __popcll(ms);
        // lane k gets the k-th source's lane (the others fill up behind)
        const int to = src ? __popcll(ms & lanemask_lt()) : nsrc + __popcll(~ms & lanemask_lt());
        const int from = __builtin_amdgcn_ds_permute(to * 4, lane);
        for (int k0 = 0; k0 < nsrc; k0 += TC_SRC * (WAVE / TC_SMALL)) {
            TcRow ru[TC_SRC], rv[TC_SRC];
            uint32_t u[TC_SRC], v[TC_SRC];
#pragma unroll
            for (int j = 0; j < TC_SRC; j++) {
                const int k = k0 + j * (WAVE / TC_SMALL) + team, l = __shfl(from, min(k, WAVE - 1), WAVE);
                ru[j] = TcRow{(uint32_t)__shfl(own.base, l, WAVE), 0u, (uint32_t)__shfl(own.n16, l, WAVE),
                              (uint32_t)__shfl(own.n32, l, WAVE)};
                u[j] = (uint32_t)(w0 + l);
                v[j] = k < nsrc && i0 + sub < ru[j].len() ? tc_entry(ru[j], i0 + sub, codes, ids, hub) : TC_PAD;
            }
#pragma unroll
            for (int j = 0; j < TC_SRC; j++) rv[j] = v[j] != TC_PAD && v[j] != u[j] ? row[v[j]] : TcRow{0u, 0u, 0u, 0u};
#pragma unroll
            for (int j = 0; j < TC_SRC; j++) {
                if (rv[j].len() == 0 || rv[j].len() > most) continue;
                const bool mine = ru[j].len() < rv[j].len();   // the source's list is the shorter one (ties: the destination's)
                const TcRow a = {mine ? ru[j].base : rv[j].base, 0u, mine ? ru[j].n16 : rv[j].n16, mine ? ru[j].n32 : rv[j].n32};
                const TcRow b = {mine ? rv[j].base : ru[j].base, 0u, mine ? rv[j].n16 : ru[j].n16, mine ? rv[j].n32 : ru[j].n32};
                const uint32_t c = tc_common(a, b, codes, ids);
                if (c && per_vertex) atomicAdd(per_vertex + (mine ? u[j] : v[j]), (unsigned long long)c);
                acc += c;
            }
        }
    }
    acc = wave_reduce_sum(acc);
    if (__lane_id() == 0 && acc) atomicAdd(&ctl->total[(blockIdx.x + threadIdx.x / WAVE) % TC_SUMS].v, (unsigned long long)acc);
}

}  // namespace

// Resolves this file's code object (see preload_code_objects in graph.hip).
void preload_tc_code() {
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&tc_hist_kernel)) != hipSuccess) (void)hipGetLastError();
}

// Counts on the stored rows (orient: on their degree orientation).  Every buffer
// is in the handle's grow-only scratch (s_tc).
static hn_status tc_run(hn_graph* g, bool orient, uint64_t* total_out, uint64_t* per_vertex, hipStream_t st) {
    const int64_t nv = g->nv, ne = g->ne;
    auto al = [](int64_t x) { return (x + 255) & ~int64_t(255); };
    if (per_vertex && nv > 0) HN_HIP(hipMemsetAsync(per_vertex, 0, sizeof(uint64_t) * (size_t)nv, st));
    if (ne == 0 || nv == 0) {
        HN_HIP(hipStreamSynchronize(st));
        *total_out = 0;
        return HN_OK;
    }
    // at most: a vertex without entries has no group, and one with a list of TC_SMALL
    // entries or fewer no task (two billion vertices with few entries need 40 bytes each)
    const int64_t groups = ne / TC_G + std::min(nv, ne) + 1;
    const int64_t tiles = groups / TC_TILE + 2;
    const int64_t tasks = std::min(nv, ne / TC_SMALL) + 2 * ne / TC_CAND + 1;
    // what an owner's stored row says of its edges holds on symmetric storage only
    const int sym = orient && graph_known_symmetric(g) ? 1 : 0;
    const uint32_t most = sym || nv <= (int64_t)TC_HUBS ? TC_SMALL : TC_SMALL_GROUPED;
    int64_t o = 0;
    auto take = [&](int64_t bytes) {
        const int64_t at = o;
        o = al(o + bytes);
        return at;
    };
    const int64_t o_ctl = take(sizeof(TcCtl)), o_hist = take(TC_BINS * 4);
    const int64_t nhub = std::min<int64_t>(nv, TC_HUBS + 1);
    const int64_t o_part = take(nhub * TC_LANES * 4), o_zero_end = o;   // cleared together
    const int64_t o_gcnt = take(nv * 4), o_weight = take(nv * 4), o_wc = take(nv * 8), o_hub = take((int64_t)(TC_HUBS + 1) * 4);
    const int64_t o_row = take(nv * (int64_t)sizeof(TcRow)), o_P = take((nv + 1) * 4), o_tile = take(tiles * 4), o_placed = take(tiles * (TC_TILE / WAVE));
    const int64_t o_codes = take(groups * TC_G * 2), o_ids = take(groups * TC_G * 4), o_place = take(groups * TC_G * 4);
    const int64_t o_goff = take((nv + 1) * 4), o_mem = take(ne * 4), o_task = take(tasks * 8);
    const int64_t bits = (nv + WAVE - 1) / WAVE * 8, o_some = take(bits), o_owner = take(bits), o_small = take(bits), o_hubs = take(bits);
    const int64_t o_scan = take((int64_t)scan_temp_bytes(nv));
    HN_TRY(g->s_tc.reserve((size_t)o));
    char* base = g->s_tc.as<char>();
    auto at = [&](int64_t off, auto* kind) { return reinterpret_cast<decltype(kind)>(base + off); };
    TcCtl* ctl = at(o_ctl, (TcCtl*)nullptr);
    uint32_t* hist = at(o_hist, (uint32_t*)nullptr);
    uint32_t* gcnt = at(o_gcnt, (uint32_t*)nullptr);
    uint32_t* part = at(o_part, (uint32_t*)nullptr);
    uint32_t* weight = at(o_weight, (uint32_t*)nullptr);
    uint2* wc = at(o_wc, (uint2*)nullptr);
    uint32_t* hub = at(o_hub, (uint32_t*)nullptr);
    TcRow* row = at(o_row, (TcRow*)nullptr);
    uint32_t* P = at(o_P, (uint32_t*)nullptr);
    uint32_t* tile_lo = at(o_tile, (uint32_t*)nullptr);
    uint16_t* codes = at(o_codes, (uint16_t*)nullptr);
    uint32_t* ids = at(o_ids, (uint32_t*)nullptr);
    uint32_t* place = at(o_place, (uint32_t*)nullptr);
    uint8_t* placed = at(o_placed, (uint8_t*)nullptr);
    uint32_t* goff = at(o_goff, (uint32_t*)nullptr);
    uint32_t* members = at(o_mem, (uint32_t*)nullptr);
    uint2* task = at(o_task, (uint2*)nullptr);
    uint64_t* some = at(o_some, (uint64_t*)nullptr);
    uint64_t* hubs = at(o_hubs, (uint64_t*)nullptr);
    uint64_t* owner = at(o_owner, (uint64_t*)nullptr);
    uint64_t* small = at(o_small, (uint64_t*)nullptr);
    void* tmp = base + o_scan;
    unsigned long long* per = reinterpret_cast<unsigned long long*>(per_vertex);
    const unsigned gv = (unsigned)ceil_div(nv, BLOCK);
    const unsigned gt = (unsigned)std::min<int64_t>(tiles, (int64_t)num_cus() * 8);
    const unsigned gw = (unsigned)std::min<int64_t>(gv, (int64_t)num_cus() * 2);

    HN_HIP(hipMemsetAsync(base, 0, (size_t)o_zero_end, st));
    // 1. hubs and codes
    const bool all_hubs = nv <= (int64_t)TC_HUBS;
    HN_TRY(exclusive_scan_fn<uint32_t>(StoredGroupsIn{g->rec},
                                       StoredGroupsOut{g->rec, row, P, tile_lo, orient && !all_hubs ? weight : nullptr, some},
                                       P + nv, nv, tmp, st));
    if (all_hubs) {
        tc_all_hubs_kernel<<<gv, BLOCK, 0, st>>>(nv, g->rec, wc, hub, ctl);
        HN_CHECK_LAUNCH();
    } else {
        if (!orient) {
            HN_HIP(hipMemsetAsync(weight, 0, (size_t)nv * 4, st));
            const int step = (int)std::clamp<int64_t>(ne >> 18, 1, 64);
            tc_weight_freq_kernel<<<gt, BLOCK, 0, st>>>(nv, P + nv, P, tile_lo, g->rec, g->arena, step, weight);
            HN_CHECK_LAUNCH();
        }
        tc_hist_kernel<<<gw, BLOCK, 0, st>>>(nv, weight, hist);
        HN_CHECK_LAUNCH();
        tc_cut_kernel<<<1, BLOCK, 0, st>>>(hist, ctl);
        HN_CHECK_LAUNCH();
        HN_TRY(exclusive_scan_fn<uint32_t>(HubIn{weight, ctl}, HubOut{weight, wc, hub, hubs}, &ctl->hubs, nv, tmp, st));
    }
    // 2. lists
    if (orient)
        tc_rows_kernel<true><<<gt, BLOCK, 0, st>>>(nv, P + nv, P, tile_lo, g->rec, g->arena, wc, nullptr, row, codes, ids, ctl);
    else
        tc_rows_kernel<false><<<gt, BLOCK, 0, st>>>(nv, P + nv, P, tile_lo, g->rec, g->arena, wc, all_hubs ? nullptr : hubs, row,
                                                    codes, ids, ctl);
    HN_CHECK_LAUNCH();
    tc_pad_kernel<<<(unsigned)ceil_div(nv, BLOCK * TC_PAD_WORDS), BLOCK, 0, st>>>(nv, some, row, codes, ids, most, owner, small, gcnt);
    HN_CHECK_LAUNCH();
    // 3. edges owned by their destination
    tc_group_kernel<false><<<gt, BLOCK, 0, st>>>(nv, P + nv, P, tile_lo, sym, ctl, row, owner, codes, ids, hub, gcnt, part, nhub,
                                                 place, placed, nullptr, nullptr);
    HN_CHECK_LAUNCH();
    tc_parts_kernel<<<(unsigned)ceil_div(nhub, BLOCK), BLOCK, 0, st>>>(sym, ctl, nhub, hub, part, gcnt);
    HN_CHECK_LAUNCH();
    HN_TRY(exclusive_scan_fn<uint64_t>(OwnerIn{owner, row, gcnt, g->rec, ctl, sym}, OwnerOut{goff, task}, &ctl->owned, nv, tmp, st));
    tc_group_kernel<true><<<gt, BLOCK, 0, st>>>(nv, P + nv, P, tile_lo, sym, ctl, row, owner, codes, ids, hub, gcnt, part, nhub,
                                                place, placed, goff, members);
    HN_CHECK_LAUNCH();
    // 4. counts
    tc_owner_kernel<<<(unsigned)num_cus() * 8, BLOCK, 0, st>>>(orient ? 1 : 0, sym, g->rec, g->arena, wc, task, row, codes, ids,
                                                               hub, gcnt, goff, members, ctl, per);
    HN_CHECK_LAUNCH();
    const int small_per = nv > TC_WIDE ? WAVE : TC_SRC * (WAVE / TC_SMALL);
    tc_small_kernel<<<(unsigned)ceil_div(nv, (int64_t)small_per * NWAVES), BLOCK, 0, st>>>(nv, small_per, most, small, row, codes, ids,
                                                                                           hub, ctl, per);
    HN_CHECK_LAUNCH();
    TcSum sums[TC_SUMS];
    HN_TRY(read_back(g, ctl->total, sizeof(sums), sums, st));
    *total_out = 0;
    for (const TcSum& x : sums) *total_out += x.v;
    return HN_OK;
}

}  // namespace hn

using namespace hn;

extern "C" {

hn_status hn_tc2_stored(hn_graph* g, uint64_t* total, uint64_t* per_vertex, void* stream) {
    HN_ARG(g && total, "null argument");
    HN_ARG(g->ne < (int64_t)0xFFFFFFFF, "edge count exceeds 32-bit queue ids");
    return tc_run(g, false, total, per_vertex, as_stream(stream));
}

hn_status hn_tc_count(hn_graph* g, uint64_t* total, uint64_t* per_vertex, void* stream) {
    HN_ARG(g && total, "null argument");
    HN_ARG(g->ne < (int64_t)0xFFFFFFFF, "edge count exceeds the 32-bit scan");
    return tc_run(g, true, total, per_vertex, as_stream(stream));
}

}  // extern "C"
