// bfs.hpp -- the single-source BFS level loop over caller-placed scratch
// (bfs.hip), shared by the entry points that own their scratch differently.
#pragma once
#include "graph.hpp"

namespace hn {

// Level-loop control on the device: the loop runs without a host round trip
// per level.  A round expands one level with the whole device (bfs_expand_kernel
// then bfs_collect_kernel); bfs_small_kernel, one workgroup, runs any number of
// levels between two rounds.  The host numbers the rounds; which level a round
// expands is data.
struct BfsRound {
    uint64_t fc;       // frontier: size << 32 | groups of four adjacency slots
    uint64_t scan;     // degree sum of the frontiers expanded before it (an estimate after
                       // bfs_small_kernel: 4 per group)
    uint64_t vis;      // sum of their sizes
    uint32_t lev;      // its level (its vertices lie at distance lev - 1)
    uint32_t prev;     // groups of the frontier before it (0: there was none)
};
struct BfsCtl {
    // round r reads rd[r % 3], adds its discoveries to rd[(r + 1) % 3].fc and
    // clears rd[(r + 2) % 3].fc for the next one: nothing that a launch reads is
    // written in it
    BfsRound rd[3];
    uint64_t claim;    // frontier slots claimed by the collect of a pull round, as in fc
    uint32_t pulled;   // whether the last round's expansion pulled, for its collect
    uint32_t pad_;
    uint32_t levels;   // last non-empty level = number of non-empty frontiers
    uint32_t rounds;   // rounds that expanded a frontier
    uint64_t visited;  // sum of the frontier sizes expanded
    uint64_t scanned;  // sum of their degrees (m_C)
    uint64_t dsum;     // sum over the expanded frontiers of size x distance
    uint64_t deg;      // degrees of the source and of bfs_small_kernel's discoveries
    uint64_t left;     // (host copy) size of the frontier that a level limit left unexpanded
};
static_assert(sizeof(BfsCtl) <= 256, "the control block keeps its place in the scratch layout");

// Scratch of one traversal, carved from one device buffer: the handle's
// s_bfs, or the static array of the no-allocation entry point.
// The frontier needs no ping-pong: collect writes each discovered vertex's
// degree, adjacency offset (in 128-byte units) and group prefix into
// (qdeg, qbase, P), and the first frontier index of every expansion tile into
// tile_lo; the next level's expansion reads them before that level's collect
// overwrites them.
constexpr int64_t BFS_ANY_BYTES = 16384;
struct BfsBufs {
    uint32_t* bitmap;   // visited as of the start of the level
    uint32_t* full;     // bit w: bitmap word w is all ones (every one of its 32 vertices visited)
    int32_t* qdeg;
    uint32_t* qbase;
    uint32_t* P;
    uint32_t* tile_lo;
    uint8_t* state;     // one byte per vertex, padded to whole bitmap words: 0 not reached, 1 .. 126 distance + 1,
                        // 127 reached, its distance is in the caller's array, 128 no edges
    uint64_t* part;     // per collect workgroup: the degrees of discoveries so far
    BfsCtl* ctl;
    uint32_t* any;      // bit b: some vertex of the b-th 2^shift is visited (BFS_ANY_BYTES)
};

// Lays the buffers of a traversal of a graph with nv vertices and ne edges
// out from `base` (nullptr: sizes only); returns the bytes they take.
int64_t bfs_layout(int64_t nv, int64_t ne, char* base, BfsBufs* b);
// BFS TopDown from `source` into dist[nv] over laid-out buffers, reading the
// level counters back through `host` (pinned, at least sizeof(BfsCtl) bytes).
// With max_levels > 0 the traversal stops after that many levels (vertices
// farther than max_levels keep INT32_MAX; the 2-hop queries of the serving
// loop); `host` then holds the traversal's last control block.  Allocates
// nothing, except the timing events when `may_time` and stats->time_kernels ask
// for kernel timing.
hn_status bfs_run(hn_graph* g, int32_t source, int32_t* dist, hn_bfs_stats* stats, hipStream_t st,
                  const BfsBufs& b, bool may_time, uint64_t* host, int32_t max_levels = 0);

}  // namespace hn
