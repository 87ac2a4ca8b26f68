// bfs.hip -- level-synchronous top-down BFS (HornetsNest BfsTopDown).
//
// Reference: hornetsnest/src/Static/BreadthFirstSearch/TopDown.cu:49-106 runs,
// per level, forAllEdges(hornet, queue, BFSOperator, BinarySearch):
// computeWorkKernel + cub ExclusiveSum + D2H total + binarySearchKernel
// (primitives/LoadBalancing/BinarySearch.i.cuh:57-101), then a queue swap with
// a <<<1,1>>> kernel and another D2H (primitives/Queue/TwoLevelQueue.i.cuh:158-179).
// Its operator is a non-atomic check-then-set (TopDown.cu:54-60), so a vertex
// may be enqueued more than once; the distances are still exact.
//
// Here no level needs the host (counts live in a device control block), and a
// level is run in one of three ways, each where it is the fastest:
//   * bfs_small_kernel, one workgroup, runs any number of levels with small
//     frontiers in one launch (the first and last levels of a skewed graph, all
//     of a road network's), and whole traversals of tiny graphs;
//   * a push round: bfs_expand_kernel marks the frontier's neighbours,
//     bfs_collect_kernel turns the marks into the next frontier;
//   * a pull round (bfs_pull), on symmetric adjacency, where the frontier holds
//     so many entries that it is cheaper to let every unreached vertex look for
//     one reached neighbour.
// Push round:
//   1. expand: the frontier arrives as (degree, adjacency offset, group
//      prefix) triples plus, per tile of the expansion, the frontier index
//      holding the tile's first group -- the partition that BinarySearchLB
//      recomputes with two global binary searches per block
//      (BinarySearchLB.i.cuh:254-264); a group is four adjacency slots (16
//      bytes).  Every edge block is a power of two of at least 32 slots and
//      128-byte aligned, so a vertex's ceil(deg/4) groups lie inside its block
//      and each is one aligned 16-byte load (slots past deg in the last group
//      are masked).  Each tile stages its frontier slice in LDS and maps a
//      group to its vertex with a fixed-step LDS search.  A neighbour in a
//      bitmap word that the LDS summary knows full was reached before the
//      level; every other one first probes the visited bitmap as of the start
//      of the level (n/8 bytes, read-only here, so L2 resident), and the
//      survivors probe the byte-per-vertex state array (0 = never reached) --
//      on levels where most of the adjacency still leads to unreached vertices
//      the bitmap probe is skipped and the state probe alone decides.  An
//      unreached neighbour is marked with an idempotent byte store: probe
//      and mark touch the same cache line, and marks made earlier in the level
//      suppress later ones.  No atomics:
//      with eight XCDs, each holding its own L2, device-scope atomics are not
//      served from cache (claiming vertices with atomicOr measured 7x slower,
//      and even XCD-private mark bitmaps with workgroup-scope atomics measured
//      1.5x slower than byte stores);
//   2. collect: a lane owns 32 vertices (32 state bytes, one word of the
//      visited bitmap as of the start of the level); a set state byte whose
//      bitmap bit is clear is a newly reached vertex: it gets its bitmap bit, so
//      every vertex enters a frontier once.  A workgroup lists its discoveries,
//      sums their degrees and groups, claims their frontier slots and group
//      range with one 64-bit atomicAdd of (count << 32 | groups), and
//      writes each discovery's triple and the tile starts inside its groups:
//      the exclusive scan of the frontier's groups that the reference runs as
//      a separate pass (cub ExclusiveSum) falls out of the slot claims.
// A pull round's expansion counts its discoveries itself; its collect folds the
// marks into the bitmap and writes the frontier only if a push comes next.
// The frontier counters rotate by round, so no launch is needed to make the
// next frontier current.  The distances are written at the end, from the state
// bytes (bfs_dist_kernel).
// R-MAT s24, one traversal: 2.3 ms with push rounds alone, 0.67 ms; s20: 0.25 ms,
// 0.14 ms; s12: 0.11 ms, 0.033 ms; a 733 x 1021 lattice from its corner: 36 ms, 4.1 ms.
// Distances: source 0, its neighbours 1, unreached INT32_MAX (TopDown.cu:42,81).
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <type_traits>

#include <hip/hip_ext.h>

#include "bfs.hpp"
#include "bfs_pulls.hpp"
#include "prims.hpp"

namespace hn {
namespace {

constexpr int EXP_G = 4;                       // adjacency slots per work unit
#ifndef BFS_EXP_IPT
#define BFS_EXP_IPT 4
#endif
#ifndef BFS_FULL_LDS_WORDS
#define BFS_FULL_LDS_WORDS 7168
#endif
#ifndef BFS_GRID_PER_CU
#define BFS_GRID_PER_CU 6    // expansion grid at most, in 256-lane workgroups per CU
#endif
#ifndef BFS_EXP_BLOCK
#define BFS_EXP_BLOCK 512
#endif
constexpr int EXP_IPT = BFS_EXP_IPT;           // work units per lane per tile
constexpr int EXP_BLOCK = BFS_EXP_BLOCK;       // expansion workgroup size
constexpr int EXP_WAVES = EXP_BLOCK / WAVE;
constexpr int EXP_TILE = EXP_BLOCK * EXP_IPT;  // work units per tile
constexpr int32_t INF = 0x7fffffff;
// The expansion keeps the first FULL_LDS_WORDS words of the full-word summary
// in LDS (28 KB: vertices below 7 * 2^20).  A neighbour whose bitmap word is known
// full was visited before the level, so its bitmap probe is skipped.  512-lane
// workgroups share one copy per 8 waves: with the 24 KB load-balancing stage,
// three workgroups fill a CU's 160 KB.
constexpr int FULL_LDS_WORDS = BFS_FULL_LDS_WORDS;
#ifndef BFS_DIRECT_OPEN_PCT
#define BFS_DIRECT_OPEN_PCT 25   // skip bitmap probes while more than this % of the adjacency volume is unreached
#endif
// The any-summary of the visited vertices (bottom-up levels): one bit per
// 2^shift vertices, 16 KB.  A collect wave covers 2,048 vertices and writes its
// bits as a whole, 16 or 8 of them; graphs above 2^25 vertices go without (0).
constexpr int ANY_WORDS = BFS_ANY_BYTES / 4;
inline int any_shift_for(int64_t nv) { return nv <= (1 << 24) ? 7 : nv <= (1 << 25) ? 8 : 0; }
static_assert(UNIT_SLOTS % EXP_G == 0, "groups must not straddle a block start");
typedef int32_t AdjVec __attribute__((ext_vector_type(EXP_G)));

// ---- one workgroup, many levels (bfs_small_kernel): up to SM_W groups
#ifndef BFS_SMALL_DENSE_W
#define BFS_SMALL_DENSE_W 1024   // ... and this many where they average more than two groups a vertex
#endif
constexpr int SM_BLOCK = 1024;
constexpr int SM_IPT = 4;                      // groups per lane in flight
constexpr uint32_t SM_DENSE_W = BFS_SMALL_DENSE_W;
constexpr int SM_CAP = 4096;                   // frontier entries held in LDS (two levels' worth, 64 KB)
constexpr int64_t SM_NE = 0xFFFF0000;          // group prefixes are kept in 30 bits
constexpr int SM_BM_WORDS = 24064;             // visited bitmap held in LDS: 94 KB, 770,048 vertices
// graphs that one launch traverses from start to end
constexpr int TINY_CAP = 8192;
constexpr int64_t TINY_NV = TINY_CAP;
constexpr int64_t TINY_NE = 1 << 18;

// State bytes: 0 not reached; 1 .. 126 reached at distance 0 .. 125;
// STATE_DIRECT reached, its distance is in the caller's array already; bit 7
// (set by pulls) no edges.  The distances of all levels but the deepest are
// written once, as whole lines, by bfs_dist_kernel at the end: written level by
// level, 4.4 M scattered distances cost 45 us of a 212 us level (R-MAT s24), and
// the array had to be filled with INT32_MAX first.
constexpr uint32_t STATE_DIRECT = 127;
constexpr uint32_t STATE_NONE = 128;
__device__ __forceinline__ uint32_t state_at(uint32_t level) { return level <= 125 ? level + 1 : STATE_DIRECT; }

// The caller's distances from the state bytes, once the traversal is over (else
// nothing, and the host launches it again).
__global__ __launch_bounds__(BLOCK) void bfs_dist_kernel(uint32_t r, int32_t max_levels, int64_t nv,
                                                         const uint8_t* __restrict__ state,
                                                         const BfsCtl* __restrict__ ctl, int32_t* __restrict__ dist) {
    const BfsRound rd = ctl->rd[r % 3];
    if ((rd.fc >> 32) != 0 && !(max_levels > 0 && (int64_t)rd.lev > max_levels)) return;
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x, nthr = (int64_t)gridDim.x * BLOCK;
    const int64_t n4 = (reinterpret_cast<uintptr_t>(dist) & 15) == 0 ? nv / 4 : 0;
    auto value = [](uint32_t b) { return (b & 127u) ? (int32_t)(b & 127u) - 1 : INF; };
    for (int64_t k = i; k < n4; k += nthr) {
        const uint32_t q = reinterpret_cast<const uint32_t*>(state)[k];
        const uint32_t d = (q & 0x7F7F7F7Fu) ^ 0x7F7F7F7Fu;   // a zero byte: STATE_DIRECT
        const uint32_t b[4] = {q & 255u, (q >> 8) & 255u, (q >> 16) & 255u, q >> 24};
        if (((d - 0x01010101u) & ~d & 0x80808080u) == 0) {
            reinterpret_cast<int4*>(dist)[k] = make_int4(value(b[0]), value(b[1]), value(b[2]), value(b[3]));
        } else {
            for (int e = 0; e < 4; e++)
                if ((b[e] & 127u) != STATE_DIRECT) dist[4 * k + e] = value(b[e]);
        }
    }
    for (int64_t k = 4 * n4 + i; k < nv; k += nthr)
        if ((state[k] & 127u) != STATE_DIRECT) dist[k] = value(state[k]);
}

__global__ void bfs_init_kernel(int32_t nv, const hn_vrec* __restrict__ rec, uint32_t* __restrict__ bitmap, uint32_t* __restrict__ full,
                                uint32_t* __restrict__ any, int any_shift, uint32_t* __restrict__ state4, int32_t source, int32_t* __restrict__ qdeg,
                                uint32_t* __restrict__ qbase, uint32_t* __restrict__ P,
                                uint32_t* __restrict__ tile_lo, uint64_t* __restrict__ part,
                                BfsCtl* __restrict__ ctl) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nthr = (int64_t)gridDim.x * blockDim.x;
    const int64_t words = ((int64_t)nv + 31) / 32;
    for (int64_t k = i; k < (words + BLOCK - 1) / BLOCK; k += nthr) part[k] = 0u;
    for (int64_t k = i; k < (words + 31) / 32; k += nthr) full[k] = 0u;
    if (any_shift > 0)
        for (int64_t k = i; k < ANY_WORDS; k += nthr)
            any[k] = k == (source >> any_shift) >> 5 ? 1u << ((source >> any_shift) & 31) : 0u;
    for (int64_t k = i; k < words; k += nthr) bitmap[k] = (k == (source >> 5)) ? (1u << (source & 31)) : 0u;
    // state bytes (4 per word, words * 8 words, 256-byte aligned): the
    // source's alone set
    for (int64_t k = i; k < words * 2; k += nthr) {
        uint4 q = make_uint4(0u, 0u, 0u, 0u);
        if (k == (source >> 4)) {
            const uint32_t b = 1u << (8 * (source & 3));
            const int o = (source >> 2) & 3;
            q.x = o == 0 ? b : 0u;
            q.y = o == 1 ? b : 0u;
            q.z = o == 2 ? b : 0u;
            q.w = o == 3 ? b : 0u;
        }
        reinterpret_cast<uint4*>(state4)[k] = q;
    }
    // the first frontier: the source alone, owning every tile of its groups
    const hn_vrec r = rec[source];
    const int64_t ng = ((int64_t)r.deg + EXP_G - 1) / EXP_G;
    for (int64_t t = i; t < (ng + EXP_TILE - 1) / EXP_TILE; t += (int64_t)gridDim.x * blockDim.x) tile_lo[t] = 0u;
    if (i == 0) {
        qdeg[0] = r.deg;
        qbase[0] = (uint32_t)(r.off / UNIT_SLOTS);
        P[0] = 0u;
        BfsCtl c{};
        c.rd[0].fc = ((uint64_t)1 << 32) | (uint64_t)ng;
        c.rd[0].lev = 1;
        c.deg = (uint64_t)r.deg;
        *ctl = c;
    }
}

// Probes go through buffer loads: a lane without a probe to make gets an
// offset past the buffer's end, which the hardware's range check answers with
// 0 and no cache access (a plain load of a shared dummy address would still
// take a cache-tag lookup in every group of four lanes that holds one).
constexpr uint32_t PROBE_NONE = 0xFFFFFFF0u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t probe_rsrc(const void* p, uint32_t bytes) {
    // raw buffer (stride 0), gfx9-family descriptor word 3
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint32_t probe_b32(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0);
}
__device__ __forceinline__ uint8_t probe_u8(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(r, (int)off, 0, 0);
}

// A round's record, known to be the same for all lanes: the rules over it run in scalar
// registers, every workgroup's first instructions.
__device__ __forceinline__ BfsRound bfs_round(const BfsRound* p) {
    BfsRound rd = *p;
    uint32_t w[sizeof(BfsRound) / 4];
    __builtin_memcpy(w, &rd, sizeof rd);
#pragma unroll
    for (uint32_t& x : w) x = (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
    __builtin_memcpy(&rd, w, sizeof rd);
    return rd;
}

// Pulling follows the stored entries backwards, so only adjacency known to be
// symmetric pulls (sym).
__device__ __forceinline__ bool bfs_pulls(const BfsRound& rd, int64_t nv, int64_t ne, int32_t sym) {
    return sym && hn::bfs_pulls(rd.fc >> 32, (uint32_t)rd.fc, rd.scan, rd.vis, nv, ne, rd.prev);
}

// the frontier slice of a tile: group prefix, adjacency offset in 128-byte
// units (every block starts on one), degree
// (LbShared sizes its stage for BLOCK threads: EXP_TILE + 1 entries)
using ExpLb = LbShared<EXP_TILE / BLOCK, uint32_t, uint32_t>;
static_assert(ExpLb::CAP == EXP_TILE + 1, "stage holds a tile's segments");
struct ExpShared {
    ExpLb lb;
    int32_t deg[ExpLb::CAP];
    uint32_t full[FULL_LDS_WORDS];     // head of the full-word summary
};

// ---- pull
#ifndef BFS_PULL_J
#define BFS_PULL_J 2
#endif
constexpr int PULL_J = BFS_PULL_J;        // open vertices per lane and batch
constexpr int PULL_BATCH = WAVE * PULL_J;
constexpr int PULL_SPAN_WORDS = 32;       // bitmap words (32 vertices each) a wave takes at a time
constexpr int PULL_SPAN_SMALL = 8;        // ... on graphs too small to give every wave that many,
// and on few words: a wave's rows that do not settle are a chain of steps (20 layers of
// 2,000 vertices with 64 edges each to the next, 510 us with 8, 400 so; R-MAT s18, whose rows do, 108 and 124 us)
constexpr int PULL_SPAN_TINY = 2;
constexpr int64_t PULL_TINY_WORDS = 2048;
constexpr int PULL_FLUSH = 112;           // rows left that make the second step run
constexpr int PULL_ROWS = PULL_FLUSH + PULL_BATCH;
constexpr int TEAM = 8;                   // lanes that scan one row: 8 x 16 bytes, a 128-byte line
constexpr int32_t WAVE_AT = 512;          // slots after which a row goes to its whole wave,
constexpr int32_t GROUP_AT = 16384;       // and to the whole workgroup
constexpr int LONG_CAP = 64;
struct PullWave {
    uint16_t open[PULL_SPAN_WORDS * 32];  // the span's unreached vertices
    uint32_t base[PULL_ROWS];             // rows that their first group did not settle: adjacency offset in 128-byte
    int32_t deg[PULL_ROWS];               // units, degree,
    uint16_t lv[PULL_ROWS];               // vertex within the span
    uint16_t lng[LONG_CAP];               // rows for the whole wave (index into the above)
};
struct PullShared {
    uint32_t any[ANY_WORDS];              // summary of the visited vertices
    PullWave w[EXP_WAVES];
    int32_t lvert[LONG_CAP];              // rows for the whole workgroup
    uint32_t nlong;
    uint64_t red[2][EXP_WAVES];
};
union StepShared {
    ExpShared push;
    PullShared pull;
};
static_assert(sizeof(StepShared) * 3 <= 160 * 1024, "three workgroups fill a CU's LDS");

struct PullSum {   // (a graph has fewer than 2^32 entries)
    uint32_t count = 0, groups = 0, degs = 0;
};

// Bottom-up expansion of one level: every vertex without its bitmap bit is
// unreached, and (the adjacency being symmetric) lies at this level iff one of
// its neighbours has its bit; the bitmap is that of the level's start and only
// read here.  Rows are ascending and skewed graphs keep their hubs at low ids,
// so most rows settle in their first 16 bytes.
// Every wave works on its own, a span of the bitmap at a time, so that its
// chain of loads (bitmap, records, first groups, probes) overlaps the other
// waves':
//   lanes: a list of the span's open vertices, then a row per lane: record and
//          first group; the rows left, listed in LDS, their next two groups (a
//          wave instruction checks 64 rows; eight lanes per row from the start
//          cost eight times the instructions: 521 against 479 us);
//   teams: of 8 lanes scan the rows left, a 128-byte line per step;
//   wave, workgroup: scan the rows left after WAVE_AT and GROUP_AT slots.
// The L1 serves one scattered probe a cycle, which bounds a level whose rows
// need many: where few vertices are visited (FILTER), a probe first asks an LDS
// summary, one bit per 2^any_shift vertices, and most end there (R-MAT s24, the
// level of 45 M frontier entries: 5 M vector memory instructions, 680 us without
// it, 447 us with it).  What bounds it then is the rate of scattered 64-byte
// reads, about 46 G/s: 8.9 M records and first row sectors alone take 230 us,
// 4.4 M 140 us (that level's next: 191 us).
// A vertex without edges is marked STATE_NONE, so that later levels skip it.
template <bool FILTER>
__device__ __forceinline__ void bfs_pull(PullShared& sh, uint32_t L, int64_t nv, int64_t words,
                                         const hn_vrec* __restrict__ rec, const int32_t* __restrict__ arena,
                                         uint8_t* __restrict__ state, const uint32_t* __restrict__ bitmap,
                                         const uint32_t* __restrict__ any, int any_shift,
                                         __amdgpu_buffer_rsrc_t rbm, int32_t* __restrict__ dist, PullSum& sum) {
    const int lane = __lane_id(), wv = threadIdx.x / WAVE;
    PullWave& W = sh.w[wv];
    if (threadIdx.x == 0) sh.nlong = 0;
    if constexpr (FILTER)
        for (int i = threadIdx.x; i < ANY_WORDS; i += EXP_BLOCK) sh.any[i] = any[i];
    __syncthreads();
    const uint8_t mark = (uint8_t)state_at(L);
    auto reach = [&](int64_t v, int32_t deg) {
        if (mark == STATE_DIRECT && dist) dist[v] = (int32_t)L;
        state[v] = mark;
        sum.count++;
        sum.groups += (uint32_t)(deg + EXP_G - 1) / EXP_G;
        sum.degs += (uint32_t)deg;
    };
    // the bitmap words of the first nval slots of x (0 where nothing is probed)
    struct Words {
        uint32_t w[EXP_G];
    };
    auto probe1 = [&](int32_t t, bool ask) {
        if constexpr (FILTER) {
            const uint32_t b = ask ? (uint32_t)t >> any_shift : 0u;
            ask = ask && ((sh.any[b >> 5] >> (b & 31)) & 1u);
        }
        return probe_b32(rbm, ask ? ((uint32_t)t >> 5) * 4u : PROBE_NONE);
    };
    auto probe = [&](const AdjVec& x, int32_t nval) {
        Words r;
#pragma unroll
        for (int e = 0; e < EXP_G; e++) r.w[e] = probe1(x[e], e < nval);
        return r;
    };
    auto hits = [&](const AdjVec& x, const Words& r) {
        uint32_t h = 0;
#pragma unroll
        for (int e = 0; e < EXP_G; e++) h |= r.w[e] >> (x[e] & 31);
        return (h & 1u) != 0;
    };
    auto load = [&](int64_t at) { return *reinterpret_cast<const AdjVec*>(arena + at); };
    // `keep` lanes' rows to the front of the list, from entry n on
    auto put = [&](int& n, bool keep, uint32_t base, int32_t deg, int lv) {
        const uint64_t m = __ballot(keep);
        if (keep) {
            const int k = n + (int)__popcll(m & lanemask_lt());
            W.base[k] = base;
            W.deg[k] = deg;
            W.lv[k] = (uint16_t)lv;
        }
        n += (int)__popcll(m);
    };
    // the n rows listed, of the span that starts at vertex v0
    auto settle = [&](int n, int64_t v0) {
        // slots 4 .. 11, two rows per lane in flight; the rows left move to the
        // front (behind the entries being read)
        int m = 0;
        for (int i0 = 0; i0 < n; i0 += 2 * WAVE) {
            uint32_t base[2];
            int32_t deg[2];
            int lv[2];
            AdjVec y[2], z[2];
            bool act[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int i = i0 + q * WAVE + lane;
                act[q] = i < n;
                base[q] = W.base[act[q] ? i : n - 1];
                deg[q] = W.deg[act[q] ? i : n - 1];
                lv[q] = W.lv[act[q] ? i : n - 1];
                y[q] = load((int64_t)base[q] * UNIT_SLOTS + EXP_G);
                z[q] = load((int64_t)base[q] * UNIT_SLOTS + 2 * EXP_G);   // (a block has 32 slots)
            }
            Words wy[2], wz[2];
#pragma unroll
            for (int q = 0; q < 2; q++) {
                wy[q] = probe(y[q], act[q] ? deg[q] - EXP_G : 0);
                wz[q] = probe(z[q], act[q] ? deg[q] - 2 * EXP_G : 0);
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const bool hit = hits(y[q], wy[q]) || hits(z[q], wz[q]);
                if (hit) reach(v0 + lv[q], deg[q]);
                put(m, act[q] && !hit && deg[q] > 3 * EXP_G, base[q], deg[q], lv[q]);
            }
            __builtin_amdgcn_wave_barrier();
        }
        // teams (the first step repeats slots 0 .. 11, to stay on whole lines)
        const int sub = lane & (TEAM - 1);
        int it = lane / TEAM, nlng = 0;
        int32_t k = 0;
        while (__ballot(it < m)) {
            const int i = it < m ? it : m - 1;
            const int32_t deg = W.deg[i];
            const int64_t row = (int64_t)W.base[i] * UNIT_SLOTS;
            const int32_t p = k + sub * EXP_G;
            const AdjVec x = load(row + (p < deg ? p : 0));
            const bool hit = hits(x, probe(x, it < m && p >= 3 * EXP_G ? deg - p : 0));
            const bool found = ((__ballot(hit) >> (lane & ~(TEAM - 1))) & ((1u << TEAM) - 1u)) != 0;
            if (found && sub == 0) reach(v0 + W.lv[i], deg);
            k += TEAM * EXP_G;
            bool next = found || k >= deg;
            // a long row goes to the wave's list (when that is full, the team goes on)
            const uint64_t lm = __ballot(it < m && !next && k >= WAVE_AT && sub == 0);
            if (lm) {
                const int q = nlng + (int)__popcll(lm & lanemask_lt());
                const bool moved = ((lm >> lane) & 1u) && q < LONG_CAP;
                if (moved) W.lng[q] = (uint16_t)it;
                next = next || ((__ballot(moved) >> (lane & ~(TEAM - 1))) & 1u);
                nlng = min(nlng + (int)__popcll(lm), LONG_CAP);
            }
            if (next) {
                it += WAVE / TEAM;
                k = 0;
            }
        }
        __builtin_amdgcn_wave_barrier();
        for (int q = 0; q < nlng; q++) {
            const int i = W.lng[q];
            const int32_t deg = W.deg[i];
            const int64_t row = (int64_t)W.base[i] * UNIT_SLOTS;
            bool found = false;
            int64_t k0 = WAVE_AT;
            while (k0 < deg && !found) {
                if (k0 >= GROUP_AT + WAVE_AT) {   // the workgroup's list, if it has room
                    uint32_t x = 0;
                    if (lane == 0) {
                        x = atomicAdd(&sh.nlong, 1u);
                        if (x < LONG_CAP) sh.lvert[x] = (int32_t)(v0 + W.lv[i]);
                        else atomicSub(&sh.nlong, 1u);
                    }
                    if ((uint32_t)__builtin_amdgcn_readfirstlane((int)x) < LONG_CAP) break;
                }
                AdjVec x[4];
                Words w[4];
#pragma unroll
                for (int h = 0; h < 4; h++) {
                    const int64_t p = k0 + (h * WAVE + lane) * EXP_G;
                    x[h] = load(row + (p < deg ? p : 0));
                }
#pragma unroll
                for (int h = 0; h < 4; h++)
                    w[h] = probe(x[h], (int32_t)min((int64_t)EXP_G, (int64_t)deg - (k0 + (h * WAVE + lane) * EXP_G)));
                bool hit = false;
#pragma unroll
                for (int h = 0; h < 4; h++) hit = hit || hits(x[h], w[h]);
                found = __ballot(hit) != 0;
                k0 += 4 * WAVE * EXP_G;
            }
            if (found && lane == 0) reach(v0 + W.lv[i], deg);
        }
    };
    // small graphs: shorter spans, so that every wave has one
    const int64_t nwaves = (int64_t)gridDim.x * EXP_WAVES;
    const int sw = words >= nwaves * PULL_SPAN_WORDS / 2 ? PULL_SPAN_WORDS
                   : words > PULL_TINY_WORDS ? PULL_SPAN_SMALL : PULL_SPAN_TINY;
    for (int64_t c = (int64_t)blockIdx.x * EXP_WAVES + wv; c * sw < words; c += nwaves) {
        const int64_t w0 = c * sw, v0 = w0 * 32;
        uint32_t bits = 0;
        if (lane < sw && w0 + lane < words) {
            bits = ~bitmap[w0 + lane];
            const int64_t left = nv - (w0 + lane) * 32;   // >= 1
            if (left < 32) bits &= (1u << left) - 1u;
        }
        const uint32_t mine = (uint32_t)__popc(bits), inc = wave_inclusive_scan(mine);
        const int n = __builtin_amdgcn_readlane((int)inc, WAVE - 1);
        if (n == 0) continue;
        for (uint32_t at = inc - mine; bits; bits &= bits - 1)
            W.open[at++] = (uint16_t)(lane * 32 + __ffs(bits) - 1);
        __builtin_amdgcn_wave_barrier();
        int nrows = 0;
        int lv[PULL_J];
        hn_vrec rv[PULL_J];
        // loads are unconditional, so that all are in flight; a lane past the
        // list's end repeats its last entry
        auto records = [&](int b0) {
#pragma unroll
            for (int j = 0; j < PULL_J; j++) {
                const int i = b0 + j * WAVE + lane;
                lv[j] = W.open[i < n ? i : n - 1];
                rv[j] = rec[v0 + lv[j]];
            }
        };
        records(0);
        for (int b0 = 0; b0 < n; b0 += PULL_BATCH) {
            AdjVec x[PULL_J];
            uint32_t unit[PULL_J];
            int32_t deg[PULL_J];
            int v[PULL_J];
#pragma unroll
            for (int j = 0; j < PULL_J; j++) {
                v[j] = lv[j];
                deg[j] = b0 + j * WAVE + lane < n ? rv[j].deg : -1;
                unit[j] = (uint32_t)(rv[j].off / UNIT_SLOTS);
                x[j] = load(rv[j].off);   // (offset 0 without a block)
            }
            if (b0 + PULL_BATCH < n) records(b0 + PULL_BATCH);   // the next batch's, while this one's rows are on their way
            // the first slot alone, then the other three where it does not
            // settle the row: late in a traversal most first slots do
            bool hit[PULL_J];
            uint32_t w0s[PULL_J];
#pragma unroll
            for (int j = 0; j < PULL_J; j++) w0s[j] = probe1(x[j][0], deg[j] > 0);
#pragma unroll
            for (int j = 0; j < PULL_J; j++) hit[j] = (w0s[j] >> (x[j][0] & 31)) & 1u;
            uint32_t w[PULL_J][EXP_G - 1];
#pragma unroll
            for (int j = 0; j < PULL_J; j++)
#pragma unroll
                for (int e = 1; e < EXP_G; e++) w[j][e - 1] = probe1(x[j][e], !hit[j] && e < deg[j]);
#pragma unroll
            for (int j = 0; j < PULL_J; j++) {
#pragma unroll
                for (int e = 1; e < EXP_G; e++) hit[j] = hit[j] || ((w[j][e - 1] >> (x[j][e] & 31)) & 1u);
                if (hit[j]) reach(v0 + v[j], deg[j]);
                if (deg[j] == 0) state[v0 + v[j]] = (uint8_t)STATE_NONE;
                put(nrows, !hit[j] && deg[j] > EXP_G, unit[j], deg[j], v[j]);
            }
            if (nrows >= PULL_FLUSH || b0 + PULL_BATCH >= n) {
                __builtin_amdgcn_wave_barrier();
                if (nrows) settle(nrows, v0);
                nrows = 0;
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    __syncthreads();
    const int nl = (int)min(sh.nlong, (uint32_t)LONG_CAP);
    for (int q = 0; q < nl; q++) {
        const int32_t v = sh.lvert[q];
        const hn_vrec rv = rec[v];
        bool found = false;
        for (int64_t k0 = GROUP_AT; k0 < rv.deg && !found; k0 += 4 * EXP_BLOCK * EXP_G) {
            bool hit = false;
#pragma unroll
            for (int h = 0; h < 4; h++) {
                const int64_t p = k0 + (h * EXP_BLOCK + (int)threadIdx.x) * EXP_G;
                const AdjVec x = load(rv.off + (p < rv.deg ? p : 0));
                hit = hits(x, probe(x, (int32_t)min((int64_t)EXP_G, (int64_t)rv.deg - p))) || hit;
            }
            found = __syncthreads_or(hit) != 0;
        }
        if (found && threadIdx.x == 0) reach(v, rv.deg);
    }
}

// One round's expansion.  Push: every neighbour of the frontier is tested against the visited bitmap and,
// if not visited before this level, against state[]; unreached ones are
// marked.  A launch marks with one value, so concurrent stores agree.
// Pull (bfs_pull): the level's discoveries are found, marked and counted here;
// the collect then only folds the marks into the bitmap.
template <int G>
__global__ __launch_bounds__(EXP_BLOCK, 6) void bfs_expand_kernel(uint32_t r, int32_t max_levels, int32_t sym, int64_t nv,
                                                           const hn_vrec* __restrict__ rec,
                                                           const uint32_t* __restrict__ P,
                                                           const uint32_t* __restrict__ tile_lo,
                                                           const int32_t* __restrict__ qdeg,
                                                           const uint32_t* __restrict__ qbase,
                                                           BfsCtl* __restrict__ ctl,
                                                           const int32_t* __restrict__ arena,
                                                           uint8_t* __restrict__ state,
                                                           const uint32_t* __restrict__ bitmap,
                                                           const uint32_t* __restrict__ full,
                                                           const uint32_t* __restrict__ any, int any_shift,
                                                           int64_t words, int64_t fwords,
                                                           uint64_t* __restrict__ part,
                                                           int64_t nparts, int64_t ne, int32_t* __restrict__ dist) {
    typedef AdjVec Vec;
    constexpr int CAP = ExpLb::CAP;
    __shared__ StepShared ssh;
    ExpShared& sh = ssh.push;
    const __amdgpu_buffer_rsrc_t rbm = probe_rsrc(bitmap, (uint32_t)(words * 4));
    const __amdgpu_buffer_rsrc_t rst = probe_rsrc(state, (uint32_t)(words * 32));
    const BfsRound rd = bfs_round(&ctl->rd[r % 3]);
    const uint32_t L = rd.lev;
    const int64_t F = (int64_t)(rd.fc >> 32);
    const bool over = F == 0 || (max_levels > 0 && (int64_t)L > max_levels);
    // round bookkeeping by workgroup 0
    if (blockIdx.x == 0) {
        if (over) {
            if (threadIdx.x == 0) {
                if (F > 0) ctl->rd[(r + 1) % 3] = rd;   // the level limit: the frontier stays as it is
                ctl->rd[(r + 2) % 3].fc = 0;
            }
        } else {
            // the degrees of every discovery so far, one partial per collect
            // workgroup, join those of the source and of the one-workgroup levels
            __shared__ uint64_t red[EXP_WAVES];
            uint64_t x = 0;
            for (int64_t i = threadIdx.x; i < nparts; i += EXP_BLOCK) x += part[i];
            x = wave_reduce_sum(x);
            if (__lane_id() == 0) red[threadIdx.x / WAVE] = x;
            __syncthreads();
            if (threadIdx.x == 0) {
                uint64_t t = ctl->deg;
                for (int k = 0; k < EXP_WAVES; k++) t += red[k];
                // (workgroups of a pull may have added discoveries to `part`
                // meanwhile: `scan` only guides bfs_pulls, and the last
                // frontier of a traversal discovers nothing)
                ctl->rd[(r + 2) % 3].fc = 0;
                ctl->rd[(r + 1) % 3].scan = t;
                ctl->rd[(r + 1) % 3].vis = rd.vis + (uint64_t)F;
                ctl->rd[(r + 1) % 3].lev = L + 1;
                ctl->rd[(r + 1) % 3].prev = (uint32_t)rd.fc;
                ctl->claim = 0;
                ctl->scanned = t;
                ctl->levels = L;
                ctl->rounds++;
                ctl->visited += (uint64_t)F;
                ctl->dsum += (uint64_t)F * (uint64_t)(L - 1);   // level L's frontier lies at distance L - 1
            }
        }
    }
    if (over) return;
    const bool pull = bfs_pulls(rd, nv, ne, sym);
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->pulled = pull ? 1u : 0u;
    if (pull) {
        PullSum s;
        // (a visited vertex sets at most one of the summary's bits)
        if (any_shift > 0 && rd.vis + (uint64_t)F < (uint64_t)ANY_WORDS * 32)
            bfs_pull<true>(ssh.pull, L, nv, words, rec, arena, state, bitmap, any, any_shift, rbm, dist, s);
        else
            bfs_pull<false>(ssh.pull, L, nv, words, rec, arena, state, bitmap, any, any_shift, rbm, dist, s);
        __syncthreads();
        const uint64_t cg = wave_reduce_sum(((uint64_t)s.count << 32) + s.groups), dg = wave_reduce_sum((uint64_t)s.degs);
        if (__lane_id() == 0) {
            ssh.pull.red[0][threadIdx.x / WAVE] = cg;
            ssh.pull.red[1][threadIdx.x / WAVE] = dg;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint64_t a = 0, d = 0;
            for (int k = 0; k < EXP_WAVES; k++) {
                a += ssh.pull.red[0][k];
                d += ssh.pull.red[1][k];
            }
            if (a) {
                atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->rd[(r + 1) % 3].fc), (unsigned long long)a);
                atomicAdd(reinterpret_cast<unsigned long long*>(part + blockIdx.x % nparts), (unsigned long long)d);
            }
        }
        return;
    }
    const int64_t W = (int64_t)(uint32_t)rd.fc;
    // Skip the bitmap probes while most adjacency entries still lead to
    // unreached vertices: the state bytes are cumulative (every vertex reached
    // so far has its byte set), so the state probe alone decides, and the
    // bitmap would only filter the few reached targets.  The share of entries
    // leading to reached vertices is estimated by the adjacency volume reached
    // before this level plus this frontier's (4 slots per group).
    const uint64_t vol = rd.scan + (uint64_t)W * G;
    const bool direct = (uint64_t)(100 - BFS_DIRECT_OPEN_PCT) * (uint64_t)ne > 100 * vol;
    const int64_t ntiles = (W + EXP_TILE - 1) / EXP_TILE;
    if ((int64_t)blockIdx.x >= ntiles) return;
    for (int i = threadIdx.x; i < FULL_LDS_WORDS; i += EXP_BLOCK) sh.full[i] = i < fwords ? full[i] : 0u;
    for (int64_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int64_t lo = tile_lo[t];
        const int64_t hi = (t + 1 < ntiles) ? (int64_t)tile_lo[t + 1] : F - 1;
        const int64_t w0 = t * EXP_TILE;
        const int64_t span = hi - lo + 1;
        const bool staged = span <= CAP;
        if (staged) {
            for (int i = threadIdx.x; i < (int)span; i += EXP_BLOCK) {
                sh.lb.pref[i] = P[lo + i];
                sh.lb.base[i] = qbase[lo + i];
                sh.deg[i] = qdeg[lo + i];
            }
        }
        __syncthreads();
        // phase 1: every unit's slot address and valid slot count
        int64_t addr[EXP_IPT];
        int nval[EXP_IPT];
        if (staged) {
#pragma unroll
            for (int j = 0; j < EXP_IPT; j++) {
                const int64_t w = w0 + (int64_t)j * EXP_BLOCK + threadIdx.x;
                const int s = lb_locate(sh.lb, (int)span, w);
                const int64_t k = (w - (int64_t)sh.lb.pref[s]) * G;
                addr[j] = (int64_t)sh.lb.base[s] * UNIT_SLOTS + k;
                nval[j] = w < W ? (int)min((int64_t)G, (int64_t)sh.deg[s] - k) : 0;
            }
        } else {   // slice wider than LDS (runs of zero-degree frontier vertices)
            for (int j = 0; j < EXP_IPT; j++) {
                const int64_t w = w0 + (int64_t)j * EXP_BLOCK + threadIdx.x;
                addr[j] = 0;
                nval[j] = 0;
                if (w < W) {
                    const int64_t s = upper_bound_m1<int64_t>(P, lo, hi + 1, w);
                    const int64_t k = (w - (int64_t)P[s]) * G;
                    addr[j] = (int64_t)qbase[s] * UNIT_SLOTS + k;
                    nval[j] = (int)min((int64_t)G, (int64_t)qdeg[s] - k);
                }
            }
        }
        // Phases 2 and 3 load unconditionally (a unit without work reads
        // arena[0..G), a slot without a probe gets an out-of-range buffer
        // offset) so that no load sits in a branch of its own, where the
        // compiler waits for it at once.
        // phase 2: all adjacency groups in flight at once (streamed, not kept in L2)
        Vec v[EXP_IPT];
#pragma unroll
        for (int j = 0; j < EXP_IPT; j++)
            v[j] = __builtin_nontemporal_load(reinterpret_cast<const Vec*>(arena + (nval[j] > 0 ? addr[j] : 0)));
        // phase 3a: all visited-bitmap probes in flight at once (n/8 bytes,
        // L2 resident), folded branch-free into one bit per candidate slot
        // (a neighbour in a word the LDS summary knows full makes no probe); on
        // direct levels the state probe alone decides
        uint32_t known = 0;
#pragma unroll
        for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
            for (int e = 0; e < G; e++) {
                const uint32_t t = e < nval[j] ? (uint32_t)v[j][e] : 0u;
                const uint32_t fw = t >> 10;
                const uint32_t f = sh.full[fw < (uint32_t)FULL_LDS_WORDS ? fw : 0u];
                known |= (uint32_t)((fw < (uint32_t)FULL_LDS_WORDS) & ((f >> ((t >> 5) & 31)) & 1u)) << (j * G + e);
            }
        uint32_t cand = 0;
        if (direct) {
#pragma unroll
            for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
                for (int e = 0; e < G; e++)
                    cand |= (uint32_t)((e < nval[j]) & !((known >> (j * G + e)) & 1u)) << (j * G + e);
        } else {
            uint32_t wb[EXP_IPT][G];
#pragma unroll
            for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
                for (int e = 0; e < G; e++)
                    wb[j][e] = probe_b32(rbm, ((e < nval[j]) && !((known >> (j * G + e)) & 1u))
                                                   ? ((uint32_t)v[j][e] >> 5) * 4u : PROBE_NONE);
#pragma unroll
            for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
                for (int e = 0; e < G; e++)
                    cand |= (uint32_t)((e < nval[j]) & !((known >> (j * G + e)) & 1u) &
                                       (((wb[j][e] >> (v[j][e] & 31)) & 1u) == 0)) << (j * G + e);
        }
        // phase 3b: candidates (not visited before this level) probe their
        // state byte; the rest make no probe
        uint8_t s[EXP_IPT][G];
#pragma unroll
        for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
            for (int e = 0; e < G; e++)
                s[j][e] = probe_u8(rst, ((cand >> (j * G + e)) & 1u) ? (uint32_t)v[j][e] : PROBE_NONE);
        uint32_t need = 0;
#pragma unroll
        for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
            for (int e = 0; e < G; e++)
                need |= (uint32_t)(((cand >> (j * G + e)) & 1u) & (s[j][e] == 0)) << (j * G + e);
        // phase 4: idempotent marks
        const uint8_t mark = (uint8_t)state_at(L);
#pragma unroll
        for (int j = 0; j < EXP_IPT; j++)
#pragma unroll
            for (int e = 0; e < G; e++)
                if (need & (1u << (j * G + e))) state[v[j][e]] = mark;
        __syncthreads();
    }
}

// One lane owns 32 vertices (32 state bytes and one visited-bitmap word):
// set state bytes not yet in the bitmap are this level's discoveries; they get
// their bitmap bit, a slot in the next frontier and a range of its groups.
// The discoveries are listed in LDS, so that neighbouring lanes read
// neighbouring records, each once: degree and offset stay in registers from
// the sums to the writes (walking the wave's words bit by bit, with the records
// read once for each, took 100 us for 4.4 M discoveries of R-MAT s24).  One
// atomic per workgroup claims slots and groups; on one address those take about
// 10 ns each, so large graphs use 1,024 lanes a workgroup (43 K discoveries of
// 16.7 M vertices: 31 us with 2,048 workgroups).
constexpr int COL_BLOCK_LARGE = 1024;
constexpr int64_t COL_LARGE_WORDS = 1 << 18;   // two workgroups of 1,024 lanes for every second CU
constexpr int COL_K = 32;      // discoveries per lane at most
template <int CB>
__global__ __launch_bounds__(CB) void bfs_collect_kernel(uint32_t r, int32_t max_levels, int32_t sym, int64_t nv,
                                                            int64_t ne, int64_t words,
                                                            const uint32_t* __restrict__ state4,
                                                            uint32_t* __restrict__ bitmap,
                                                            uint32_t* __restrict__ full, uint32_t* __restrict__ any,
                                                            int any_shift, int32_t* __restrict__ dist,
                                                            const hn_vrec* __restrict__ rec,
                                                            int32_t* __restrict__ qdeg, uint32_t* __restrict__ qbase,
                                                            uint32_t* __restrict__ P, uint32_t* __restrict__ tile_lo,
                                                            uint64_t* __restrict__ part, BfsCtl* __restrict__ ctl) {
    const BfsRound rd = bfs_round(&ctl->rd[r % 3]);
    if ((rd.fc >> 32) == 0) return;   // a round launched after the traversal ended
    if (max_levels > 0 && (int64_t)rd.lev > max_levels) return;
    const int32_t level = (int32_t)rd.lev;
    // after a pull the discoveries are counted; their frontier is written only if
    // the next round pushes it
    const bool pulled = __builtin_amdgcn_readfirstlane((int)ctl->pulled) != 0;
    const bool want_list = !pulled || !bfs_pulls(bfs_round(&ctl->rd[(r + 1) % 3]), nv, ne, sym);
    const int64_t wi = (int64_t)blockIdx.x * CB + threadIdx.x;
    uint32_t found = 0;
    bool wfull = false, wany = false;
    if (wi < words) {
        const uint4* p = reinterpret_cast<const uint4*>(state4 + wi * 8);
        const uint4 a = p[0], b = p[1];
        const uint32_t m[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t set = 0, none = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            // byte j of word k is vertex 32*wi + 4k + j: bits 0, 8, 16, 24 of
            // each word move to bits 0..3
            const uint32_t low = ((m[k] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) >> 7;   // bit 0 of a byte: its low 7 bits are not 0
            set |= (((low & 0x01010101u) * 0x01020408u) >> 24) << (4 * k);
            none |= ((((m[k] >> 7) & 0x01010101u) * 0x01020408u) >> 24) << (4 * k);
        }
        if (set | none) {
            const uint32_t old = bitmap[wi];
            found = set & ~old;
            // a vertex without edges is no one's neighbour: its bit only keeps
            // later pulls from looking at it
            const uint32_t now = old | found | none;
            if (now != old) bitmap[wi] = now;
        }
        // state bytes are never cleared during a traversal, so `set` is every
        // vertex of the word visited so far: the word is full iff all are
        // (or have no edges)
        wfull = (set | none) == 0xFFFFFFFFu;
        wany = set != 0;
    }
    {
        // the full-word summary: a wave owns 64 consecutive words = 2 summary words
        const uint64_t fb = __ballot(wfull);
        const int64_t fw = (wi - __lane_id()) >> 5;
        if (__lane_id() == 0 && fb && fw < (words + 31) / 32) full[fw] = (uint32_t)fb;
        if (__lane_id() == 1 && (fb >> 32) && fw + 1 < (words + 31) / 32) full[fw + 1] = (uint32_t)(fb >> 32);
    }
    if (any_shift > 0) {
        // the wave's 2,048 vertices as bits of 2^any_shift: 4 or 8 words each
        uint64_t ab = __ballot(wany);
        ab |= ab >> 1;
        ab |= ab >> 2;   // bit 4k: any of words 4k .. 4k + 3
        if (any_shift == 8) ab |= ab >> 4;
        const int64_t wv = wi - __lane_id();
        if (wv < words) {
            const int lane = __lane_id();
            const int step = any_shift == 8 ? 8 : 4;
            const uint64_t bits = __ballot(lane < 64 / step && ((ab >> (lane * step)) & 1u));
            if (lane == 0) {
                if (any_shift == 8) reinterpret_cast<uint8_t*>(any)[wv / 64] = (uint8_t)bits;
                else reinterpret_cast<uint16_t*>(any)[wv / 64] = (uint16_t)bits;
            }
        }
    }
    if (!want_list) return;
    constexpr int CW = CB / WAVE;
    constexpr int COL_CHUNK = CB > BLOCK ? 4 : 8;   // records in flight per lane
    __shared__ uint16_t list[CB * 32];      // vertex within the workgroup's CB * 32
    __shared__ uint32_t wcnt[CW];
    __shared__ uint64_t wsum[CW], went[CW], bslot;
    const int lane = __lane_id(), w = threadIdx.x / WAVE;
    const uint32_t mine = (uint32_t)__popc(found), inc = wave_inclusive_scan(mine);
    if (lane == WAVE - 1) wcnt[w] = inc;
    __syncthreads();
    uint32_t n = 0, at = inc - mine;
#pragma unroll
    for (int k = 0; k < CW; k++) {
        at += k < w ? wcnt[k] : 0u;
        n += wcnt[k];
    }
    if (n == 0) return;
    for (; found; found &= found - 1) list[at++] = (uint16_t)(threadIdx.x * 32 + __ffs(found) - 1);
    __syncthreads();
    // wave w takes entries [i0, i1) of the list, lane l every 64th
    const uint32_t share = (n + CB - 1) / CB * WAVE;
    const uint32_t i0 = min(n, w * share), i1 = min(n, i0 + share);
    const int64_t v0 = (int64_t)blockIdx.x * CB * 32;
    int32_t deg[COL_K];
    uint32_t unit[COL_K];
    uint32_t cg = 0;
    uint64_t ce = 0;
#pragma unroll
    for (int k0 = 0; k0 < COL_K; k0 += COL_CHUNK) {
        if (i0 + k0 * WAVE >= i1) break;
        hn_vrec rv[COL_CHUNK];
#pragma unroll
        for (int k = 0; k < COL_CHUNK; k++) rv[k] = rec[v0 + list[min(i0 + (k0 + k) * WAVE + lane, i1 - 1)]];
#pragma unroll
        for (int k = 0; k < COL_CHUNK; k++) {
            deg[k0 + k] = i0 + (k0 + k) * WAVE + lane < i1 ? rv[k].deg : 0;
            unit[k0 + k] = (uint32_t)(rv[k].off / UNIT_SLOTS);
            cg += ((uint32_t)deg[k0 + k] + EXP_G - 1) / EXP_G;
            ce += (uint32_t)deg[k0 + k];
        }
    }
    cg = wave_reduce_sum(cg);
    ce = wave_reduce_sum(ce);
    if (lane == 0) {
        wsum[w] = cg;
        went[w] = ce;
    }
    __syncthreads();
    // One atomicAdd per workgroup claims its frontier slots and groups
    // (count << 32 | groups: a level's groups stay below 2^32, so the low half
    // never carries); their entries add to the workgroup's own partial.
    if (threadIdx.x == 0) {
        uint64_t acc = (uint64_t)n << 32, acce = 0;
        for (int k = 0; k < CW; k++) {
            acc += wsum[k];
            acce += went[k];
        }
        uint64_t* claim = pulled ? &ctl->claim : &ctl->rd[(r + 1) % 3].fc;
        bslot = atomicAdd(reinterpret_cast<unsigned long long*>(claim), (unsigned long long)acc);
        if (!pulled) part[blockIdx.x] += acce;
    }
    __syncthreads();
    const uint32_t s0 = (uint32_t)(bslot >> 32);
    uint32_t gb = (uint32_t)bslot;
    for (int k = 0; k < w; k++) gb += (uint32_t)wsum[k];
    const bool direct = dist && state_at((uint32_t)level) == STATE_DIRECT && !pulled;
#pragma unroll
    for (int k = 0; k < COL_K; k++) {
        const uint32_t i = i0 + k * WAVE + lane;
        if (i0 + k * WAVE >= i1) break;
        const uint32_t ng = ((uint32_t)deg[k] + EXP_G - 1) / EXP_G;
        const uint32_t sc = wave_inclusive_scan(ng);
        if (i < i1) {
            const uint64_t g0 = (uint64_t)gb + sc - ng;
            if (direct) dist[v0 + list[i]] = level;
            qdeg[s0 + i] = deg[k];
            qbase[s0 + i] = unit[k];
            P[s0 + i] = (uint32_t)g0;
            for (uint64_t t = (g0 + EXP_TILE - 1) / EXP_TILE; t * EXP_TILE < g0 + ng; t++) tile_lo[t] = s0 + i;
        }
        gb += (uint32_t)__builtin_amdgcn_readlane((int)sc, WAVE - 1);
    }
}

// ---------------------------------------------------------------- one workgroup
// Levels whose frontier holds at most SM_W groups and SM_CAP vertices, by one
// workgroup in one launch: frontier in LDS, and the visited bitmap too where
// nv allows (else it is claimed in L2, with workgroup-scope atomics: nothing
// else runs on it).  A level is a chain of two loads, the adjacency group and
// the record of each newly claimed neighbour, and one barrier, where a round
// of two whole-device launches takes over 10 us however small the frontier.
// 733 x 1021 lattice, from its corner 1,753 levels of up to 733 vertices: 36 ms with
// one round per level, 4.1 ms so, 2.3 us a level: two loads from memory; from its middle
// 877 levels of up to 1,466: 21 ms, 3.9 ms.  It stops where the frontier outgrows it,
// and leaves everything as a round would: state bytes, bitmap, frontier arrays, counters.
// INIT: the whole traversal of a graph with at most TINY_NV vertices and
// TINY_NE entries (frontiers of any size fit), in this launch alone.
// A workgroup barrier that orders LDS only: __syncthreads also waits until the
// level's stores to memory are acknowledged, which nothing in the level loop
// reads.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int CAP, int BMW, int ANYW>
struct SmallShared {
    uint2 ent[2][CAP];       // x: group prefix << 2 | deg % 4, y: adjacency offset in 128-byte units
    uint32_t bm[BMW];
    uint32_t any[ANYW];      // the summary, where the bitmap is in memory
    uint32_t bm0[BMW > TINY_NV / 32 ? 1 : BMW];   // one-launch pulls: the level's start
    unsigned long long cnt[3];   // per level % 3: size << 32 | groups
    uint32_t multi[3];           // some vertex of the level has other than one group
    uint64_t red[2][SM_BLOCK / WAVE];
    uint32_t ntodo, nlong;       // one-launch pulls
    uint32_t lrow[LONG_CAP];
};

// One-launch pulls: most of a small skewed graph is reached in one level whose
// frontier holds most of its entries (R-MAT s12: 20 K groups, 40 us as a push
// with its claims, against about 4 us).
// Returns this lane's discoveries through `append`, called by whole waves.
template <typename Append>
__device__ __forceinline__ void bfs_tiny_pull(int nv, const hn_vrec* __restrict__ rec,
                                              const int32_t* __restrict__ arena, const uint32_t* __restrict__ bm,
                                              uint2* __restrict__ todo, uint32_t* ntodo, uint32_t* nlong,
                                              uint32_t* lrow, Append append) {
    const int tid = threadIdx.x, lane = __lane_id();
    auto hit_any = [&](const AdjVec& x, int nval) {
        bool hit = false;
#pragma unroll
        for (int e = 0; e < EXP_G; e++) {
            const uint32_t t = e < nval ? (uint32_t)x[e] : 0u;
            hit = hit || (e < nval && ((bm[t >> 5] >> (t & 31)) & 1u));
        }
        return hit;
    };
    // as bfs_pull's phases: a lane per vertex, a team per row left, the workgroup
    constexpr int J = 4;
    for (int v0 = 0; v0 < nv; v0 += SM_BLOCK * J) {
        bool open[J];
        hn_vrec rv[J];
        AdjVec a[J];
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int v = v0 + j * SM_BLOCK + tid;
            open[j] = v < nv && !((bm[(v < nv ? v : 0) >> 5] >> (v & 31)) & 1u);
            rv[j] = rec[v < nv ? v : nv - 1];
        }
#pragma unroll
        for (int j = 0; j < J; j++) a[j] = *reinterpret_cast<const AdjVec*>(arena + (open[j] ? rv[j].off : 0));
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int v = v0 + j * SM_BLOCK + tid;
            const bool hit = hit_any(a[j], open[j] ? rv[j].deg : 0);
            append(hit, v, rv[j]);
            if (open[j] && !hit && rv[j].deg > EXP_G)
                todo[atomicAdd(ntodo, 1u)] =
                    make_uint2((uint32_t)v | ((uint32_t)rv[j].deg << 13), (uint32_t)(rv[j].off / UNIT_SLOTS));
        }
    }
    __syncthreads();
    const int n = (int)*ntodo;
    const int sub = lane & (TEAM - 1);
    int it = tid / TEAM;
    uint2 e = todo[it < n ? it : 0];
    int k = 0;
    while (__ballot(it < n)) {
        const int deg = it < n ? (int)(e.x >> 13) : 0;
        const int p = k + sub * EXP_G;
        const int64_t row = (int64_t)e.y * UNIT_SLOTS;
        const AdjVec x = *reinterpret_cast<const AdjVec*>(arena + (it < n ? row + (p < deg ? p : 0) : 0));
        const bool found = ((__ballot(hit_any(x, deg - p)) >> (lane & ~(TEAM - 1))) & ((1u << TEAM) - 1u)) != 0;
        k += TEAM * EXP_G;
        bool next = found || k >= deg;
        if (!next && sub == 0 && k >= 512) {
            const uint32_t q = atomicAdd(nlong, 1u);
            if (q < LONG_CAP) {
                lrow[q] = (uint32_t)it;
                next = true;
            } else {
                atomicSub(nlong, 1u);
            }
        }
        hn_vrec rv;
        rv.off = row;
        rv.deg = deg;
        append(found && sub == 0, (int)(e.x & 8191u), rv);
        next = __shfl((int)next, lane & ~(TEAM - 1), WAVE) != 0;
        if (next) {
            it += SM_BLOCK / TEAM;
            k = 0;
            if (it < n) e = todo[it];
        }
    }
    __syncthreads();
    const int nl = (int)min(*nlong, (uint32_t)LONG_CAP);
    for (int q = 0; q < nl; q++) {
        const uint2 f = todo[lrow[q]];
        hn_vrec rv;
        rv.off = (int64_t)f.y * UNIT_SLOTS;
        rv.deg = (int32_t)(f.x >> 13);
        bool found = false;
        for (int k0 = 512; k0 < rv.deg && !found; k0 += SM_BLOCK * EXP_G) {
            const int p = k0 + tid * EXP_G;
            const AdjVec x = *reinterpret_cast<const AdjVec*>(arena + rv.off + (p < rv.deg ? p : 0));
            found = __syncthreads_or(hit_any(x, rv.deg - p)) != 0;
        }
        append(found && tid == 0, (int)(f.x & 8191u), rv);
    }
}

template <int CAP, int BMW, bool LDSBM, bool INIT>
__global__ __launch_bounds__(SM_BLOCK) void bfs_small_kernel(uint32_t r, int32_t max_levels, int32_t sym, int64_t nv,
                                                             int64_t ne, int32_t source,
                                                             const hn_vrec* __restrict__ rec,
                                                             const int32_t* __restrict__ arena,
                                                             int32_t* __restrict__ dist, uint8_t* __restrict__ state,
                                                             uint32_t* bitmap, uint32_t* any, int any_shift,
                                                             int64_t words, int32_t* __restrict__ qdeg, uint32_t* __restrict__ qbase,
                                                             uint32_t* __restrict__ P, uint32_t* __restrict__ tile_lo,
                                                             const uint64_t* __restrict__ part, int64_t nparts,
                                                             BfsCtl* __restrict__ ctl, BfsCtl* __restrict__ host,
                                                             int first) {
    __shared__ SmallShared<CAP, BMW, LDSBM ? 1 : ANY_WORDS> sh;
    const int tid = threadIdx.x, lane = __lane_id();
    BfsRound rd{};
    uint64_t visited = 0, scanned = 0, dsum = 0, deg = 0;
    uint32_t levels = 0, rounds = 0;
    if constexpr (INIT) {
        const hn_vrec sr = rec[source];
        rd.fc = (1ull << 32) | (uint32_t)((sr.deg + EXP_G - 1) / EXP_G);
        rd.lev = 1;
        deg = (uint64_t)sr.deg;
        if (dist)
            for (int64_t v = tid; v < nv; v += SM_BLOCK) dist[v] = v == source ? 0 : INF;
        for (int i = tid; i < (int)words; i += SM_BLOCK) sh.bm[i] = i == (source >> 5) ? 1u << (source & 31) : 0u;
        if (tid == 0) sh.ent[1][0] = make_uint2((uint32_t)sr.deg & 3u, (uint32_t)(sr.off / UNIT_SLOTS));
    } else {
        rd = ctl->rd[r % 3];
        visited = ctl->visited;
        scanned = ctl->scanned;
        dsum = ctl->dsum;
        deg = ctl->deg;
        levels = ctl->levels;
        rounds = ctl->rounds;
    }
    uint32_t L = rd.lev;
    uint64_t fc = rd.fc;
    auto fits = [&]() {
        return (fc >> 32) != 0 && !(max_levels > 0 && (int64_t)L > max_levels) &&
               (INIT || ((fc >> 32) <= (uint64_t)CAP && ne < SM_NE &&
                         ((uint32_t)fc <= SM_DENSE_W || ((uint32_t)fc <= SM_W && (uint32_t)fc <= 2 * (fc >> 32)))));
    };
    const bool work = fits();
    uint64_t degs = 0;             // degrees of the discoveries
    if (work) {
        if constexpr (!INIT) {
            const int F = (int)(fc >> 32);
            for (int i = tid; i < F; i += SM_BLOCK)
                sh.ent[L & 1][i] = make_uint2((P[i] << 2) | ((uint32_t)qdeg[i] & 3u), qbase[i]);
            if constexpr (LDSBM) {
                for (int i = tid; i < (int)words; i += SM_BLOCK) sh.bm[i] = first ? 0u : bitmap[i];
                if (first && tid == (source >> 5) % SM_BLOCK) sh.bm[source >> 5] = 1u << (source & 31);
            } else if (any_shift > 0) {
                const uint32_t ab = (uint32_t)source >> any_shift;
                for (int i = tid; i < ANY_WORDS; i += SM_BLOCK)
                    sh.any[i] = !first ? any[i] : i == (int)(ab >> 5) ? 1u << (ab & 31) : 0u;
            }
        }
        if (tid < 3) {
            sh.cnt[tid] = 0;
            sh.multi[tid] = 1;   // the first level searches; the others' flags are cleared before their use
            if (tid == (int)((L + 1) % 3)) sh.multi[tid] = 0;
            if (tid == (int)((L + 2) % 3)) sh.multi[tid] = 0;
        }
        __syncthreads();
    }
    while (fits()) {
        const uint32_t F = (uint32_t)(fc >> 32), W = (uint32_t)fc;
        const uint2* cur = sh.ent[L & 1];
        uint2* nxt = sh.ent[(L + 1) & 1];
        const bool multi = sh.multi[L % 3] != 0;
        levels = L;
        visited += F;
        dsum += (uint64_t)F * (L - 1);
        rd.scan += 4ull * W;
        rd.vis += F;
        const uint32_t prev = rd.prev;
        rd.prev = W;
        const int top = 31 - __clz((int)F | 1);   // F < 2^(top + 1)
        // a claimed vertex's distance, and its frontier entry
        auto mark = [&](int32_t v) {
            if (dist) dist[v] = (int32_t)L;
            if constexpr (!LDSBM) {   // (else from the bitmap at the end)
                state[v] = (uint8_t)STATE_DIRECT;
                // (in LDS: neighbouring ids share a word, and atomics on one word in memory take 10 ns each)
                const uint32_t ab = (uint32_t)v >> any_shift;
                if (any_shift > 0) atomicOr(&sh.any[ab >> 5], 1u << (ab & 31));
            }
        };
        auto found = [&](int32_t v, const hn_vrec& rv, uint32_t slot, uint32_t gb) {
            const uint32_t base = (uint32_t)(rv.off / UNIT_SLOTS);
            mark(v);
            if (slot < (uint32_t)CAP) {
                nxt[slot] = make_uint2((gb << 2) | ((uint32_t)rv.deg & 3u), base);
            } else if constexpr (!INIT) {   // the frontier outgrows LDS: a round takes it
                const uint32_t ng = (uint32_t)(rv.deg + EXP_G - 1) / EXP_G;
                qdeg[slot] = rv.deg;
                qbase[slot] = base;
                P[slot] = gb;
                for (uint64_t t = ((uint64_t)gb + EXP_TILE - 1) / EXP_TILE; t * EXP_TILE < (uint64_t)gb + ng; t++)
                    tile_lo[t] = slot;
            }
        };
        // a vertex won: its slot, groups and counters (wave-wide)
        auto append = [&](bool won, int v, const hn_vrec& rv) {
            if (__ballot(won) == 0) return;
            const uint32_t ng = won ? (uint32_t)(rv.deg + EXP_G - 1) / EXP_G : 0u;
            const uint32_t ic = wave_inclusive_scan(won ? 1u : 0u), ig = wave_inclusive_scan(ng);
            unsigned long long b = 0;
            if (lane == WAVE - 1) b = atomicAdd(&sh.cnt[(L + 1) % 3], ((unsigned long long)ic << 32) | ig);
            const uint32_t slot = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), WAVE - 1) + ic - 1;
            const uint32_t g0 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, WAVE - 1) + ig - ng;
            if (won) {
                nxt[slot] = make_uint2((g0 << 2) | ((uint32_t)rv.deg & 3u), (uint32_t)(rv.off / UNIT_SLOTS));
                atomicOr(&sh.bm[v >> 5], 1u << (v & 31));
                if (dist) dist[v] = (int32_t)L;
                degs += (uint32_t)rv.deg;
                sh.multi[(L + 1) % 3] = 1;
            }
        };
        // every unreached vertex costs a pull at least one group, and one that it does not
        // reach (see bfs_pulls) all of its row: 20 layers of 300 vertices with 16 edges each
        // to the next, 380 us without, 130 so
        const uint64_t open = (uint64_t)nv - visited, mu = (uint64_t)ne > rd.scan ? (uint64_t)ne - rd.scan : 0;
        const bool pull = INIT && sym && W > SM_DENSE_W && 2 * (uint64_t)W > open &&
                          (2 * (uint64_t)W > open + mu / EXP_G || 2 * (uint64_t)W > open + bfs_wasted(F, W, prev, open, mu) / EXP_G);
        if constexpr (INIT)
            if (pull) {
                for (int i = tid; i < (int)words; i += SM_BLOCK) sh.bm0[i] = sh.bm[i];
                if (tid == 0) sh.ntodo = sh.nlong = 0;
                __syncthreads();
                // the frontier's own list is not needed any more: the rows left go there
                bfs_tiny_pull((int)nv, rec, arena, sh.bm0, sh.ent[L & 1], &sh.ntodo, &sh.nlong, sh.lrow, append);
            }
        // Every frontier vertex has one group (roads, paths): a lane per slot,
        // NJ of them in flight, without a branch per lane: nothing searches, and
        // the claims and record loads of a wave overlap (6.3 -> 5.4 ms).
        auto slots = [&](auto njc, uint32_t i0) {
            constexpr int NJ = decltype(njc)::value;
            int32_t t[NJ];
            uint32_t bit[NJ], old[NJ], word[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const uint32_t i = i0 + j * SM_BLOCK + lane, s = i / EXP_G, e = i % EXP_G;
                const uint2 en = cur[min(s, F - 1)];
                bit[j] = s < F && ((en.x & 3u) == 0 || e < (en.x & 3u)) ? 1u : 0u;
                t[j] = arena[(int64_t)en.y * UNIT_SLOTS + e];   // (a block has 32 slots)
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                // claim: the one lane that sets a vertex's bit owns the discovery
                // (a lane without a slot sets no bit of word 0, in LDS; in memory that
                // many atomics on one word took 10 ns each: a binary tree of a million
                // vertices 540 us with them, 360 so)
                word[j] = bit[j] ? (uint32_t)t[j] >> 5 : 0u;
                bit[j] <<= t[j] & 31;
                if constexpr (LDSBM) old[j] = atomicOr(&sh.bm[word[j]], bit[j]);
                else old[j] = bit[j] ? __hip_atomic_fetch_or(bitmap + word[j], bit[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) : 0u;
            }
            bool won[NJ];
            hn_vrec rv[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                won[j] = (bit[j] & ~old[j]) != 0;
                rv[j] = rec[won[j] ? t[j] : 0];
            }
            uint32_t cc = 0, cg = 0;
            bool other = false;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const uint32_t d = won[j] ? (uint32_t)rv[j].deg : 0u;
                cc += won[j] ? 1u : 0u;
                cg += (d + EXP_G - 1) / EXP_G;
                degs += d;
                other = other || (won[j] && d - 1 >= (uint32_t)EXP_G);
            }
            const uint32_t ic = wave_inclusive_scan(cc);
            const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)ic, WAVE - 1);
            if (all == 0) return;
            const bool mixed = __ballot(other) != 0;
            const uint32_t ig = mixed ? wave_inclusive_scan(cg) : ic;
            unsigned long long b = 0;
            if (lane == WAVE - 1) b = atomicAdd(&sh.cnt[(L + 1) % 3], ((unsigned long long)ic << 32) | ig);
            if (mixed) sh.multi[(L + 1) % 3] = 1;
            const uint32_t sb = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), WAVE - 1);
            uint32_t slot = sb + ic - cc;
            uint32_t gb = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, WAVE - 1) + ig - cg;
            const bool fit = sb + all <= (uint32_t)CAP;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                if (won[j]) {
                    if (fit) {
                        mark(t[j]);
                        nxt[slot] = make_uint2((gb << 2) | ((uint32_t)rv[j].deg & 3u), (uint32_t)(rv[j].off / UNIT_SLOTS));
                    } else {
                        found(t[j], rv[j], slot, gb);
                    }
                    slot++;
                    gb += (uint32_t)(rv[j].deg + EXP_G - 1) / EXP_G;
                }
            }
        };
        if (!multi && !pull) {
            const uint32_t S = 4 * F;
            for (uint32_t i0 = (uint32_t)__builtin_amdgcn_readfirstlane(tid); i0 < S; i0 += SM_BLOCK * SM_IPT) {
                const uint32_t nj = (S - i0 + SM_BLOCK - 1) / SM_BLOCK;   // of this wave
                if (nj == 1) slots(std::integral_constant<int, 1>(), i0);
                else if (nj == 2) slots(std::integral_constant<int, 2>(), i0);
                else if (nj == 3) slots(std::integral_constant<int, 3>(), i0);
                else slots(std::integral_constant<int, SM_IPT>(), i0);
            }
        }
        // every lane of a wave runs every step: the appends are wave-wide
        for (uint32_t u0 = 0; u0 + (tid - lane) < W && multi && !pull; u0 += SM_BLOCK * SM_IPT) {
            const int nj = (int)min((uint32_t)SM_IPT, (W - u0 - (tid - lane) + SM_BLOCK - 1) / SM_BLOCK);
            AdjVec a[SM_IPT];
            int nval[SM_IPT];
#pragma unroll
            for (int j = 0; j < SM_IPT; j++) {
                nval[j] = 0;
                if (j >= nj) break;
                const uint32_t u = u0 + j * SM_BLOCK + tid;
                int64_t at = 0;
                if (u < W) {
                    uint32_t s = 0;   // the largest s with prefix <= u
                    for (int b = top; b >= 0; b--) {
                        const uint32_t q = s + (1u << b);
                        s = (q < F && (cur[min(q, F - 1)].x >> 2) <= u) ? q : s;
                    }
                    const uint2 e = cur[s];
                    const uint32_t k = u - (e.x >> 2);
                    const uint32_t end = s + 1 < F ? cur[s + 1].x >> 2 : W;
                    nval[j] = (u + 1 == end && (e.x & 3u)) ? (int)(e.x & 3u) : EXP_G;
                    at = (int64_t)e.y * UNIT_SLOTS + (int64_t)k * EXP_G;
                }
                a[j] = *reinterpret_cast<const AdjVec*>(arena + at);
            }
#pragma unroll
            for (int j = 0; j < SM_IPT; j++) {
                if (j >= nj) break;
                // claim: the one lane that sets a vertex's bit owns the discovery
                uint32_t won = 0;
#pragma unroll
                for (int e = 0; e < EXP_G; e++)
                    if (e < nval[j]) {
                        const uint32_t t = (uint32_t)a[j][e], bit = 1u << (t & 31);
                        if constexpr (LDSBM) {
                            if (!(sh.bm[t >> 5] & bit)) won |= (atomicOr(&sh.bm[t >> 5], bit) & bit) ? 0u : 1u << e;
                        } else {
                            // a stale set bit cannot be: bits are never cleared
                            if (!(bitmap[t >> 5] & bit))
                                won |= (__hip_atomic_fetch_or(bitmap + (t >> 5), bit, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_WORKGROUP) & bit) ? 0u : 1u << e;
                        }
                    }
                if (__ballot(won != 0) == 0) continue;
                hn_vrec rv[EXP_G];
#pragma unroll
                for (int e = 0; e < EXP_G; e++) rv[e] = rec[(won >> e) & 1u ? a[j][e] : 0];
                uint32_t cc = 0, cg = 0;
                bool other = false;
#pragma unroll
                for (int e = 0; e < EXP_G; e++)
                    if ((won >> e) & 1u) {
                        const uint32_t ng = (uint32_t)(rv[e].deg + EXP_G - 1) / EXP_G;
                        cc++;
                        cg += ng;
                        other = other || ng != 1;
                        degs += (uint32_t)rv[e].deg;
                    }
                const uint32_t ic = wave_inclusive_scan(cc), ig = wave_inclusive_scan(cg);
                unsigned long long b = 0;
                if (lane == WAVE - 1) b = atomicAdd(&sh.cnt[(L + 1) % 3], ((unsigned long long)ic << 32) | ig);
                const uint32_t sb = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), WAVE - 1) + ic - cc;
                uint32_t gb = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, WAVE - 1) + ig - cg;
                if (other) sh.multi[(L + 1) % 3] = 1;   // every writer stores the same value
                uint32_t slot = sb;
#pragma unroll
                for (int e = 0; e < EXP_G; e++)
                    if ((won >> e) & 1u) {
                        found(a[j][e], rv[e], slot, gb);
                        slot++;
                        gb += (uint32_t)(rv[e].deg + EXP_G - 1) / EXP_G;
                    }
            }
        }
        // counters of three levels rotate, so that one barrier a level is enough:
        // the next level's are read, those after it were cleared a level ago, and
        // this level's are cleared for the level after those
        lds_barrier();
        L++;
        const unsigned long long x = sh.cnt[L % 3];
        fc = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)) << 32) |
             (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
        if (tid == 0) {
            sh.cnt[(L + 2) % 3] = 0;
            sh.multi[(L + 2) % 3] = 0;
        }
    }
    __syncthreads();
    const bool over = (fc >> 32) == 0 || (max_levels > 0 && (int64_t)L > max_levels);
    if constexpr (!INIT && LDSBM)
        if (work && (dist || !over)) {
            // the state bytes of the vertices claimed here, and their bits
            for (int i = tid; i < (int)words; i += SM_BLOCK) {
                const uint32_t was = first ? (i == (source >> 5) ? 1u << (source & 31) : 0u) : bitmap[i];
                const uint32_t now = sh.bm[i], won = now & ~was;
                if (!won) continue;
                uint4* q = reinterpret_cast<uint4*>(state + (int64_t)i * 32);
                uint4 a = q[0], b = q[1];
                // four bits of a word to the low bits of four bytes
                auto bytes = [&](int k) { return ((((won >> (4 * k)) & 15u) * 0x00204081u) & 0x01010101u) * STATE_DIRECT; };
                a.x |= bytes(0), a.y |= bytes(1), a.z |= bytes(2), a.w |= bytes(3);
                b.x |= bytes(4), b.y |= bytes(5), b.z |= bytes(6), b.w |= bytes(7);
                q[0] = a;
                q[1] = b;
                bitmap[i] = now;
            }
        }
    // A round takes over: the frontier and the summary.  (A traversal that is over needs
    // neither: from a vertex without edges, R-MAT s16 39 us with them, 30 so.)
    if constexpr (!INIT)
        if (work && !over) {
            const uint32_t F = (uint32_t)(fc >> 32), W = (uint32_t)fc;
            const uint32_t n = min(F, (uint32_t)CAP);
            const uint2* cur = sh.ent[L & 1];
            for (uint32_t i = tid; i < n; i += SM_BLOCK) {
                const uint2 e = cur[i];
                const uint64_t g0 = e.x >> 2;
                const uint64_t g1 = i + 1 < n ? cur[i + 1].x >> 2 : F > n ? P[n] : W;
                qdeg[i] = (int32_t)((g1 - g0) * EXP_G - ((e.x & 3u) ? EXP_G - (e.x & 3u) : 0u));
                qbase[i] = e.y;
                P[i] = (uint32_t)g0;
                for (uint64_t t = (g0 + EXP_TILE - 1) / EXP_TILE; t * EXP_TILE < g1; t++) tile_lo[t] = i;
            }
            if constexpr (LDSBM) {
                // a lane per bit, of four words (any_shift is 7 here)
                // (a vertex without edges may set one: nothing probes it)
                for (int b0 = tid - lane; b0 * 4 < (int)words; b0 += SM_BLOCK) {
                    uint32_t x = 0;
                    for (int k = 0; k < 4; k++) {
                        const int w = (b0 + lane) * 4 + k;
                        x |= w < (int)words ? sh.bm[w] : 0u;
                    }
                    const uint64_t bits = __ballot(x != 0);
                    if (lane == 0) any[b0 / 32] = (uint32_t)bits;
                    if (lane == 1) any[b0 / 32 + 1] = (uint32_t)(bits >> 32);
                }
            } else if (any_shift > 0) {
                for (int i = tid; i < ANY_WORDS; i += SM_BLOCK) any[i] = sh.any[i];
            }
        }
    // the degree sums (and, when the traversal is over after whole-device
    // rounds, those of their discoveries)
    uint64_t x = 0;
    if (!INIT && over && work && rounds)
        for (int64_t i = tid; i < nparts; i += SM_BLOCK) x += part[i];
    const uint64_t s0 = wave_reduce_sum(degs), s1 = wave_reduce_sum(x);
    if (lane == 0) {
        sh.red[0][tid / WAVE] = s0;
        sh.red[1][tid / WAVE] = s1;
    }
    __syncthreads();
    if (tid == 0) {
        uint64_t parts = 0;
        for (int k = 0; k < SM_BLOCK / WAVE; k++) {
            deg += sh.red[0][k];
            parts += sh.red[1][k];
        }
        rd.fc = fc;
        rd.lev = L;
        if (work) scanned = deg + parts;
        for (BfsCtl* p : {INIT ? nullptr : work ? ctl : nullptr, host}) {   // host: pinned, read once the stream is done
            if (!p) continue;
            p->rd[r % 3] = rd;
            p->visited = visited;
            p->scanned = scanned;
            p->dsum = dsum;
            p->deg = deg;
            p->levels = levels;
            p->rounds = rounds;
        }
    }
}

}  // namespace

// Resolves this file's code object (see preload_code_objects in graph.hip).
void preload_bfs_code() {
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&bfs_init_kernel)) != hipSuccess) (void)hipGetLastError();
}

// Lays the buffers of a traversal of a graph with nv vertices and ne edges
// out from `base` (nullptr: sizes only); returns the bytes they take.
int64_t bfs_layout(int64_t nv_in, int64_t ne, char* base, BfsBufs* b) {
    const int64_t nv = nv_in > 0 ? nv_in : 1;
    const int64_t words = (nv + 31) / 32;
    const int64_t tiles = (ne / EXP_G + nv) / EXP_TILE + 2;
    auto al = [](int64_t x) { return (x + 255) & ~int64_t(255); };
    const int64_t o_bitmap = 0;
    const int64_t o_full = al(o_bitmap + words * 4);
    const int64_t o_qdeg = al(o_full + (words + 31) / 32 * 4);
    const int64_t o_qbase = al(o_qdeg + nv * 4);
    const int64_t o_P = al(o_qbase + nv * 4);
    const int64_t o_tile = al(o_P + nv * 4);
    const int64_t o_state = al(o_tile + tiles * 4);
    const int64_t o_part = al(o_state + words * 32);
    const int64_t o_ctl = al(o_part + ceil_div(words, BLOCK) * 8);
    const int64_t o_any = al(o_ctl + (int64_t)sizeof(BfsCtl));
    const int64_t total = o_any + BFS_ANY_BYTES;
    if (base) {
        b->bitmap = reinterpret_cast<uint32_t*>(base + o_bitmap);
        b->full = reinterpret_cast<uint32_t*>(base + o_full);
        b->qdeg = reinterpret_cast<int32_t*>(base + o_qdeg);
        b->qbase = reinterpret_cast<uint32_t*>(base + o_qbase);
        b->P = reinterpret_cast<uint32_t*>(base + o_P);
        b->tile_lo = reinterpret_cast<uint32_t*>(base + o_tile);
        b->state = reinterpret_cast<uint8_t*>(base + o_state);
        b->part = reinterpret_cast<uint64_t*>(base + o_part);
        b->ctl = reinterpret_cast<BfsCtl*>(base + o_ctl);
        b->any = reinterpret_cast<uint32_t*>(base + o_any);
    }
    return total;
}

// The level loop over laid-out buffers.  A tiny graph is one launch.  Otherwise
// the host queues the one-workgroup kernel, then as many whole-device rounds as
// the last traversal of this graph took (three before the first), then the
// one-workgroup kernel again (if there was a round), which takes the tail and writes
// the control block to the host's pinned memory; if the traversal is not over by then, 1, 2, 4,
// ... rounds more, each time followed by the one-workgroup kernel.  Rounds
// queued past the end change nothing.  Nothing here allocates (kernel timing,
// which creates its events, only with `may_time`).
hn_status bfs_run(hn_graph* g, int32_t source, int32_t* dist, hn_bfs_stats* stats, hipStream_t st,
                  const BfsBufs& b, bool may_time, uint64_t* host, int32_t max_levels) {
    const int64_t nv = g->nv, ne = g->ne;
    const int64_t words = (nv + 31) / 32;
    const int64_t nparts = ceil_div(words, BLOCK);
    // frontier adjacency offsets are kept in 128-byte units as 32-bit words
    // (2^32 units = 512 GiB of arena, more than one device holds)
    HN_ARG(g->cap_units < ((int64_t)1 << 32), "edge arena beyond 2^32 128-byte units");
    const int32_t sym = graph_known_symmetric(g) ? 1 : 0;
    const int any_shift = any_shift_for(nv);
    BfsCtl* hctl = reinterpret_cast<BfsCtl*>(host);
    const bool timed = may_time && stats && stats->time_kernels;
    // kernel timing: one event pair around each expanding launch of a chunk
    constexpr int MAX_LAUNCH = hn_graph::BFS_EVENTS / 2;
    constexpr int64_t MAX_ROUNDS = MAX_LAUNCH - 2;   // and the one-workgroup launches before and after
    hipEvent_t* ev = g->bfs_ev;
    if (timed)
        for (int i = 0; i < 2 * MAX_LAUNCH; i++)
            if (!ev[i] && hipEventCreate(&ev[i]) != hipSuccess) {
                (void)hipGetLastError();
                ev[i] = nullptr;
                set_error("bfs: event creation failed");
                return HN_E_HIP;
            }
    int nev = 0;   // event pairs recorded in this chunk
    hipError_t e = hipSuccess;
    // timed: the events take the dispatch's own start and end
    // (hipExtLaunchKernel), with no marker between the launches
#define BFS_LAUNCH(kernel, grid, block, ...)                                                             \
    do {                                                                                                 \
        if (timed)                                                                                       \
            hipExtLaunchKernelGGL(kernel, dim3((unsigned)(grid)), dim3(block), 0, st, ev[2 * nev],       \
                                  ev[2 * nev + 1], 0, __VA_ARGS__);                                      \
        else                                                                                             \
            hipLaunchKernelGGL(kernel, dim3((unsigned)(grid)), dim3(block), 0, st, __VA_ARGS__);         \
        nev++;                                                                                           \
        e = hipGetLastError();                                                                           \
    } while (0)
    const int64_t grid = std::min<int64_t>((int64_t)num_cus() * BFS_GRID_PER_CU * BLOCK / EXP_BLOCK,
                                           std::max(ceil_div(ne / EXP_G + nv, EXP_TILE), ceil_div(words, (words > PULL_TINY_WORDS ? PULL_SPAN_SMALL : PULL_SPAN_TINY) * EXP_WAVES)));
    uint32_t r = 0;   // rounds launched
    const bool tiny = nv <= TINY_NV && ne <= TINY_NE;
    auto small = [&](int first) {
        if (tiny)
            BFS_LAUNCH((bfs_small_kernel<TINY_CAP, TINY_NV / 32, true, true>), 1, SM_BLOCK, r, max_levels, sym, nv, ne,
                       source, g->rec, g->arena, dist, b.state, b.bitmap, b.any, any_shift, words, b.qdeg, b.qbase, b.P, b.tile_lo,
                       b.part, nparts, b.ctl, hctl, first);
        else if (words <= SM_BM_WORDS)
            BFS_LAUNCH((bfs_small_kernel<SM_CAP, SM_BM_WORDS, true, false>), 1, SM_BLOCK, r, max_levels, sym, nv, ne,
                       source, g->rec, g->arena, dist, b.state, b.bitmap, b.any, any_shift, words, b.qdeg, b.qbase, b.P, b.tile_lo,
                       b.part, nparts, b.ctl, hctl, first);
        else
            BFS_LAUNCH((bfs_small_kernel<SM_CAP, 1, false, false>), 1, SM_BLOCK, r, max_levels, sym, nv, ne, source,
                       g->rec, g->arena, dist, b.state, b.bitmap, b.any, any_shift, words, b.qdeg, b.qbase, b.P, b.tile_lo, b.part,
                       nparts, b.ctl, hctl, first);
    };
    if (!tiny) {
        // kernels only (no memset node), so a captured copy of this sequence replays correctly
        bfs_init_kernel<<<(unsigned)std::min<int64_t>(ceil_div(nv, BLOCK * 8), 4096), BLOCK, 0, st>>>(
            g->nv, g->rec, b.bitmap, b.full, b.any, any_shift, reinterpret_cast<uint32_t*>(b.state), source, b.qdeg, b.qbase, b.P,
            b.tile_lo, b.part, b.ctl);
        HN_CHECK_LAUNCH();
        small(1);
        if (e != hipSuccess) {
            set_error(std::string("bfs launch: ") + hipGetErrorString(e));
            return HN_E_HIP;
        }
    }
    const int last = g->bfs_last_rounds.load(std::memory_order_relaxed);
    int64_t next = tiny ? 0 : std::min<int64_t>(last >= 0 ? last : 3, MAX_ROUNDS);
    if (max_levels > 0) next = std::min<int64_t>(next, max_levels);
    int64_t ramp = 1, kns = 0;
    for (;;) {
        for (int64_t k = 0; k < next && e == hipSuccess; k++) {
            BFS_LAUNCH(bfs_expand_kernel<EXP_G>, grid, EXP_BLOCK, r, max_levels, sym, nv, g->rec, b.P, b.tile_lo,
                       b.qdeg, b.qbase, b.ctl, g->arena, b.state, b.bitmap, b.full, b.any, any_shift, words, (words + 31) / 32, b.part,
                       nparts, ne, dist);
            if (e != hipSuccess) break;
            if (words >= COL_LARGE_WORDS)
                bfs_collect_kernel<COL_BLOCK_LARGE>
                    <<<(unsigned)ceil_div(words, COL_BLOCK_LARGE), COL_BLOCK_LARGE, 0, st>>>(
                        r, max_levels, sym, nv, ne, words, reinterpret_cast<const uint32_t*>(b.state), b.bitmap,
                        b.full, b.any, any_shift, dist, g->rec, b.qdeg, b.qbase, b.P, b.tile_lo, b.part, b.ctl);
            else
                bfs_collect_kernel<BLOCK><<<(unsigned)nparts, BLOCK, 0, st>>>(
                    r, max_levels, sym, nv, ne, words, reinterpret_cast<const uint32_t*>(b.state), b.bitmap, b.full,
                    b.any, any_shift, dist, g->rec, b.qdeg, b.qbase, b.P, b.tile_lo, b.part, b.ctl);
            e = hipGetLastError();
            r++;
        }
        // (without rounds since the last one it would find nothing to do)
        if (e == hipSuccess && (next > 0 || tiny)) small(0);
        if (e == hipSuccess && dist && !tiny) {
            bfs_dist_kernel<<<(unsigned)std::min<int64_t>(ceil_div(nv, BLOCK * 8), 4096), BLOCK, 0, st>>>(
                r, max_levels, nv, b.state, b.ctl, dist);
            e = hipGetLastError();
        }
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (timed && e == hipSuccess)
            for (int k = 0; k < nev && e == hipSuccess; k++) {
                float ms = 0.f;
                e = hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]);
                kns += (int64_t)((double)ms * 1e6);
            }
        nev = 0;
        if (e != hipSuccess) {
            set_error(std::string("bfs level: ") + hipGetErrorString(e));
            return HN_E_HIP;
        }
        // done: the next frontier is empty, or the level limit is reached
        const BfsRound& rd = hctl->rd[r % 3];
        if ((rd.fc >> 32) == 0 || (max_levels > 0 && (int64_t)rd.lev > max_levels)) break;
        if ((int64_t)r > nv + 64) {   // cannot happen: every round reaches a new vertex
            set_error("bfs: level loop did not end");
            return HN_E_HIP;
        }
        next = ramp;
        ramp = std::min<int64_t>(2 * ramp, 16);
    }
#undef BFS_LAUNCH
    // the next full traversal queues as many rounds as this one needed
    if (max_levels <= 0 && !tiny) g->bfs_last_rounds.store((int)hctl->rounds, std::memory_order_relaxed);
    hctl->left = hctl->rd[r % 3].fc >> 32;
    if (stats) {
        stats->levels = (int32_t)hctl->levels;
        stats->visited = (int64_t)hctl->visited;
        stats->edges_scanned = (int64_t)hctl->scanned;
        stats->expand_ns = kns;
        stats->expand_launches = (int32_t)hctl->levels;
        stats->pad_ = 0;
    }
    return HN_OK;
}

}  // namespace hn

using namespace hn;

extern "C" hn_status hn_bfs_topdown(hn_graph* g, int32_t source, int32_t* dist, hn_bfs_stats* stats,
                                    void* stream) {
    HN_ARG(g && dist, "null argument");
    HN_ARG(source >= 0 && source < g->nv, "source outside [0, nv)");
    HN_ARG(g->ne < (int64_t)0xFFFFFFFF, "edge count exceeds the 32-bit work prefix");
    BfsBufs b;
    HN_TRY(g->s_bfs.reserve((size_t)bfs_layout(g->nv, g->ne, nullptr, &b)));
    bfs_layout(g->nv, g->ne, g->s_bfs.as<char>(), &b);
    return bfs_run(g, source, dist, stats, as_stream(stream), b, true, g->h_pinned);
}


// ---------------------------------------------------------------------------
// BFS TopDown without allocation, for callers that cannot allocate (code under
// HIP graph capture, tight serving loops).  Its traversal scratch is one
// static device array per GPU, held until the process ends; its device address
// is looked up once per device with hipGetSymbolAddress, and only that address
// is handed to kernels (the array's name is a host-side stand-in).  Every call
// on a GPU shares that GPU's array: calls that overlap on one GPU race.
// ---------------------------------------------------------------------------
namespace hn {
namespace {

constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(64) << 20;
constexpr int NOALLOC_MAX_DEVICES = 64;

// (the any-summary comes on top of the limit)
__device__ __align__(256) char scratch[NOALLOC_SCRATCH_BYTES + BFS_ANY_BYTES];

std::mutex g_scratch_mu;
char* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};

// The current device's copy of `scratch`, looked up on its first use.
hn_status noalloc_scratch(char** out) {
    int dev = -1;
    HN_HIP(hipGetDevice(&dev));
    HN_ARG(dev >= 0 && dev < NOALLOC_MAX_DEVICES, "device ordinal beyond the no-allocation table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error(std::string("no-allocation scratch: hipGetSymbolAddress: ") + hipGetErrorString(e));
            return HN_E_HIP;
        }
        g_scratch_ptr[dev] = static_cast<char*>(p);
    }
    *out = g_scratch_ptr[dev];
    return HN_OK;
}

}  // namespace
}  // namespace hn

extern "C" hn_status hn_bfs_topdown_noalloc_limit(int64_t* scratch_bytes) {
    HN_ARG(scratch_bytes, "null argument");
    *scratch_bytes = (int64_t)NOALLOC_SCRATCH_BYTES;
    return HN_OK;
}

extern "C" hn_status hn_bfs_topdown_noalloc(hn_graph* g, int32_t source, int32_t* dist, hn_bfs_stats* stats,
                                            void* stream) {
    HN_ARG(g && dist, "null argument");
    HN_ARG(source >= 0 && source < g->nv, "source outside [0, nv)");
    HN_ARG(g->ne < (int64_t)0xFFFFFFFF, "edge count exceeds the 32-bit work prefix");
    BfsBufs b;
    const int64_t need = bfs_layout(g->nv, g->ne, nullptr, &b) - BFS_ANY_BYTES;
    if (need > (int64_t)NOALLOC_SCRATCH_BYTES) {
        set_error("hn_bfs_topdown_noalloc: the graph needs " + std::to_string(need) +
                  " bytes of traversal scratch, more than the static " +
                  std::to_string(NOALLOC_SCRATCH_BYTES) + " (use hn_bfs_topdown)");
        return HN_E_CAPACITY;
    }
    char* base = nullptr;
    HN_TRY(noalloc_scratch(&base));
    bfs_layout(g->nv, g->ne, base, &b);
    return bfs_run(g, source, dist, stats, as_stream(stream), b, false, g->h_pinned);
}
