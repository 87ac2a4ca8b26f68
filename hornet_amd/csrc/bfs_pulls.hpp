// bfs_pulls.hpp -- when a BFS round pulls (plain C++: the CPU tests build it too)
#pragma once
#include <cstdint>

namespace hn {

// Groups of a frontier that one workgroup expands: no round pulls fewer.
#ifndef BFS_SMALL_W
#define BFS_SMALL_W 4096
#endif
constexpr uint32_t SM_W = BFS_SMALL_W;

// x / d within 4 %, d > 0, by the highest five bits of d (the reciprocals of 16.5 / 16 to
// 31.5 / 16 in 256ths): divisions take a round 0.7 us.
constexpr uint64_t bfs_quotient(uint64_t x, uint64_t d) {
    const int k = 63 - __builtin_clzll(d);
    const int i = (int)((k >= 4 ? d >> (k - 4) : d << (4 - k)) & 15u);
    const uint64_t r = (i < 8 ? 0xaeb6bfc8d2ddeaf8ull : 0x82868b90959ba1a7ull) >> (8 * (i & 7)) & 255u;
    const uint64_t q = x >> k;
    return q < (uint64_t)1 << 48 ? q * r >> 8 : q;
}
// Of `open` unreached vertices, whose rows hold `mu` slots, those that a frontier of `size`
// vertices and W groups, discovered from one of `prev` groups, will reach, and the slots
// of the others.
constexpr uint64_t bfs_found(uint64_t size, uint32_t W, uint32_t prev, uint64_t open) {
    const uint64_t most = 4 * (uint64_t)W < open ? 4 * (uint64_t)W : open;
    if (size * W >= most * prev) return most;   // (products below 2^63; so too where nothing is known)
    const uint64_t like = bfs_quotient(size * W, prev);
    return like < most ? like : most;
}
constexpr uint64_t bfs_wasted(uint64_t size, uint32_t W, uint32_t prev, uint64_t open, uint64_t mu) {
    const uint64_t left = prev > 0 ? open - bfs_found(size, W, prev, open) : 0;
    return left > 0 ? bfs_quotient(mu * left, open) : 0;
}

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
// That holds where the entries of unreached vertices lead anywhere.  Where a level's
// vertices know those of a few levels around them only (layers, meshes), most open
// vertices read their whole row for nothing.  So what the frontier will discover is
// estimated by what the one before it did, of `prev` groups (0: not known): as many per
// group, `size` / prev; and a slot of the rows that stay open costs a pull what an entry
// costs a push (20 layers of 600, 2,000 and 20,000 vertices with 16 edges each to the
// next: 360, 420, 505 us with push rounds of an earlier form, 790, 815, 855 without this
// estimate, 325, 385, 475 with it).
// The expansion asks, and the collect before it does: one that finds the next round
// pulling writes no frontier for it: they must agree.  So the rule is in whole
// numbers, which every copy of it evaluates alike (a sum of products in floating point
// may be contracted differently in each kernel).
constexpr bool bfs_pulls(uint64_t size, uint32_t W, uint64_t scan, uint64_t vis, int64_t nv, int64_t ne, uint32_t prev = 0) {
    if (W <= SM_W) return false;
    const int64_t mf = 4 * (int64_t)W;                                             // < 2^34
    const int64_t mu = ne > (int64_t)scan + mf ? ne - (int64_t)scan - mf : 0;      // < 2^32
    const int64_t nu = nv - (int64_t)vis - (int64_t)size;                          // < 2^31
    const int64_t touch = nu < mu ? nu : mu;
    // (the most that it can be)
    if (7 * mf + 20 * (mf < touch ? mf : touch) <= 4 * nv + 16 * touch) return false;
    const int64_t found = (int64_t)bfs_found(size, W, prev, (uint64_t)touch);
    const int64_t wasted = (int64_t)bfs_wasted(size, W, prev, (uint64_t)touch, (uint64_t)mu);
    const int64_t gain = 7 * mf + 20 * found - 4 * nv - 16 * touch - 7 * wasted;
    // half of min(mu, touch * ne / mf) < gain
    return gain > 0 && (mu < 2 * gain || (unsigned __int128)((uint64_t)touch * (uint64_t)ne) <
                                             (unsigned __int128)(2 * (uint64_t)gain) * (uint64_t)mf);
}

}  // namespace hn
