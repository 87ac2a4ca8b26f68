// bfs_pulls.hpp -- when a BFS round pulls (plain C++: the CPU tests build it too)
#pragma once
#include <cstdint>

namespace hn {

// Groups of a frontier that one workgroup expands: no round pulls fewer.
#ifndef BFS_SMALL_W
#define BFS_SMALL_W 4096
#endif
constexpr uint32_t SM_W = BFS_SMALL_W;

// Whether a round over a frontier of `size` vertices and W groups pulls (every unreached
// vertex looks for a reached neighbour) instead of pushing (every frontier vertex
// marks its neighbours); scan, vis: entries and vertices of the frontiers before it.
// Estimated device time in ps: a push takes about 7 per frontier entry
// and 20 per discovery, whose frontier entry the collect writes (R-MAT s24: 45 M
// entries, 4.4 M discoveries, 320 + 100 us); a pull reads every record (4 per
// vertex) and the first line of every unreached vertex with edges (25; about
// half of an R-MAT's vertices have none, which the first pull finds out, so 16
// per vertex not reached), and ne / (frontier entries) slots of each on average
// before it meets the frontier, fewer in skewed graphs, whose rows begin with
// the hubs (0.5 per slot).
// The expansion and the collect both ask, and a collect that finds the next round
// pulling writes no frontier for it: they must agree.  So the rule is in whole
// numbers, which every copy of it evaluates alike (a sum of products in floating point
// may be contracted differently in each kernel).
constexpr bool bfs_pulls(uint64_t size, uint32_t W, uint64_t scan, uint64_t vis, int64_t nv, int64_t ne) {
    if (W <= SM_W) return false;
    const int64_t mf = 4 * (int64_t)W;                                             // < 2^34
    const int64_t mu = ne > (int64_t)scan + mf ? ne - (int64_t)scan - mf : 0;      // < 2^32
    const int64_t nu = nv - (int64_t)vis - (int64_t)size;                          // < 2^31
    const int64_t touch = nu < mu ? nu : mu;
    const int64_t gain = 7 * mf + 20 * (mf < touch ? mf : touch) - 4 * nv - 16 * touch;
    // half of min(mu, touch * ne / mf) < gain
    return gain > 0 && (mu < 2 * gain || (unsigned __int128)((uint64_t)touch * (uint64_t)ne) <
                                             (unsigned __int128)(2 * (uint64_t)gain) * (uint64_t)mf);
}

}  // namespace hn
