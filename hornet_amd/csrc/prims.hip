// prims.hip -- wave64 LSD radix sort of 64-bit keys (optionally with a 32-bit
// value per key).
//
// Replaces the lexicographic (src,dst) batch sort of the reference, two stable
// thrust::sort_by_key calls (hornet/include/Core/SoA/impl/SoAPtr.i.cuh:560-571),
// with one sort of packed (src << bits | dst) keys.  Each pass: per-tile digit
// histogram in LDS, a scan of the digit-major histogram, then a stable scatter
// that ranks keys with 8 ballots per digit (one per digit bit, 64-lane
// ballots) and stages the tile in LDS in digit order so that global writes
// come out as per-bucket runs.
#include "prims.hpp"

#include <algorithm>
#include <utility>

namespace hn {

// ------------------------------------------------------------------ radix sort
namespace {

constexpr int RS_BITS = 8;
constexpr int RS_BUCKETS = 1 << RS_BITS;

// A pass over tiles of THREADS * IPT keys, IPT consecutive rows of 64 to a wave:
// counts per tile and digit, their prefix per digit, and the scatter.
//
// Tiles are handed out so that neighbours run on one XCD (workgroups go round the
// XCDS XCDs): a digit's runs of neighbouring tiles adjoin, and the line that they
// share is put together in one L2 instead of being written in part from two.  67 M
// keys (6 passes of 1.6 GB): scatter 410 us without, 227 with (4.7 TB/s), which the
// rows of counts (39 -> 24 us) and the counting (150 -> 140) now follow.
constexpr int XCDS = 8;
__device__ __forceinline__ int64_t rs_tile(int64_t ntiles) {
    const int64_t x = blockIdx.x % XCDS, i = blockIdx.x / XCDS;
    const int64_t each = ntiles / XCDS, more = ntiles % XCDS;   // XCD x has each + (x < more) tiles
    return x * each + min(x, more) + i;
}

template <int THREADS, int IPT>
__global__ __launch_bounds__(THREADS) void rs_hist_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                          int shift, int64_t ntiles,
                                                          uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[RS_BUCKETS];
    if (threadIdx.x < RS_BUCKETS) cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (THREADS * IPT);
    uint64_t k[IPT];
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const int64_t i = base + (int64_t)j * THREADS + threadIdx.x;
        k[j] = i < n ? keys[i] : 0;
    }
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const int64_t i = base + (int64_t)j * THREADS + threadIdx.x;
        if (i < n) atomicAdd(&cnt[(k[j] >> shift) & (RS_BUCKETS - 1)], 1u);
    }
    __syncthreads();
    if (threadIdx.x < RS_BUCKETS) hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];
}

// Per digit (one workgroup each): exclusive prefix of its per-tile counts
// across the tiles, and the digit's total.  The scatter adds the digit's start
// (prefix of the totals over smaller digits), so a pass needs no global scan.
constexpr int RS_SCAN_IPT = 8;
__global__ __launch_bounds__(BLOCK) void rs_rowscan_kernel(const uint32_t* __restrict__ hist, int64_t ntiles,
                                                           uint32_t* __restrict__ hoff, uint32_t* __restrict__ dtot) {
    __shared__ uint32_t sc[NWAVES + 1];
    const uint32_t* row = hist + (int64_t)blockIdx.x * ntiles;
    uint32_t* out = hoff + (int64_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (int64_t t0 = 0; t0 < ntiles; t0 += BLOCK * RS_SCAN_IPT) {
        // a lane's values are consecutive
        const int64_t t = t0 + threadIdx.x * RS_SCAN_IPT;
        uint32_t x[RS_SCAN_IPT], sum = 0;
#pragma unroll
        for (int j = 0; j < RS_SCAN_IPT; j++) x[j] = t + j < ntiles ? row[t + j] : 0u;
#pragma unroll
        for (int j = 0; j < RS_SCAN_IPT; j++) sum += x[j];
        uint32_t tot;
        uint32_t at = carry + block_exclusive_scan(sum, sc, &tot);
#pragma unroll
        for (int j = 0; j < RS_SCAN_IPT; j++) {
            if (t + j < ntiles) out[t + j] = at;
            at += x[j];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) dtot[blockIdx.x] = carry;
}

// exclusive prefix over the digits of one value per digit thread (the others call too)
template <int THREADS>
__device__ __forceinline__ uint32_t rs_digit_scan(uint32_t x, uint32_t* wtot) {
    const uint32_t inc = wave_inclusive_scan(x);
    if (__lane_id() == WAVE - 1 && threadIdx.x < RS_BUCKETS) wtot[threadIdx.x / WAVE] = inc;
    __syncthreads();
    uint32_t at = inc - x;
    for (int q = 0; q < (int)(threadIdx.x / WAVE) && q < RS_BUCKETS / WAVE; q++) at += wtot[q];
    __syncthreads();
    return at;
}

// KV: a 32-bit value rides with each key (staged beside it in LDS)
template <bool KV, int THREADS, int IPT>
__global__ __launch_bounds__(THREADS) void rs_scatter_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                             int shift, int64_t ntiles,
                                                             const uint32_t* __restrict__ hoff,
                                                             const uint32_t* __restrict__ dtot,
                                                             uint64_t* __restrict__ out,
                                                             const uint32_t* __restrict__ vin,
                                                             uint32_t* __restrict__ vout) {
    constexpr int TILE = THREADS * IPT, WAVES = THREADS / WAVE;
    __shared__ uint32_t wcnt[WAVES][RS_BUCKETS];    // per-wave digit counts, then starts within the tile
    __shared__ uint32_t gbase[RS_BUCKETS];          // global start of the tile's digit run, less its start in the tile
    __shared__ uint64_t stage[TILE];
    __shared__ uint32_t vstage[KV ? TILE : 1];
    __shared__ uint32_t wtot[RS_BUCKETS / WAVE];

    const int w = threadIdx.x / WAVE;
    const int l = __lane_id();
    const int64_t tile = rs_tile(ntiles);
    for (int d = threadIdx.x; d < WAVES * RS_BUCKETS; d += THREADS) (&wcnt[0][0])[d] = 0;

    const int64_t base = tile * TILE + (int64_t)w * WAVE * IPT;
    uint64_t k[IPT];
    uint32_t v[IPT], rank[IPT];
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const int64_t i = base + (int64_t)j * WAVE + l;
        k[j] = i < n ? keys[i] : 0;
        if constexpr (KV) v[j] = i < n ? vin[i] : 0;
    }
    // (the digits' totals and the tile's offsets, on their way meanwhile)
    uint32_t total = 0, before_tile = 0;
    if (threadIdx.x < RS_BUCKETS) {
        total = dtot[threadIdx.x];
        before_tile = hoff[(int64_t)threadIdx.x * ntiles + tile];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const bool valid = base + (int64_t)j * WAVE + l < n;
        const uint32_t d = (uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < RS_BITS; b++) {
            const uint64_t bal = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t before = (uint32_t)__popcll(peers & lt);
        const uint32_t start = valid ? wcnt[w][d] : 0;
        rank[j] = start + before;
        // the lowest peer lane publishes the new count after every peer has read it
        if (valid && before == 0) wcnt[w][d] = start + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    // per digit: totals over waves, then starts
    uint32_t run = 0;
    if (threadIdx.x < RS_BUCKETS) {
#pragma unroll
        for (int q = 0; q < WAVES; q++) run += wcnt[q][threadIdx.x];
    }
    const uint32_t first = rs_digit_scan<THREADS>(run, wtot);
    // digit d starts after every key of the smaller digits
    const uint32_t dbase = rs_digit_scan<THREADS>(total, wtot);
    if (threadIdx.x < RS_BUCKETS) {
        gbase[threadIdx.x] = dbase + before_tile - first;
        uint32_t at = first;
#pragma unroll
        for (int q = 0; q < WAVES; q++) {
            const uint32_t c = wcnt[q][threadIdx.x];
            wcnt[q][threadIdx.x] = at;
            at += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        if (base + (int64_t)j * WAVE + l < n) {
            const uint32_t p = wcnt[w][(uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1)] + rank[j];
            stage[p] = k[j];
            if constexpr (KV) vstage[p] = v[j];
        }
    }
    __syncthreads();
    const int tile_n = (int)min((int64_t)TILE, n - tile * TILE);
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const int p = j * THREADS + threadIdx.x;
        if (p < tile_n) {
            const uint64_t key = stage[p];
            // (32-bit wrap-around: gbase may lie below the run's start in the tile)
            const uint32_t at = gbase[(uint32_t)(key >> shift) & (RS_BUCKETS - 1)] + (uint32_t)p;
            out[at] = key;
            if constexpr (KV) vout[at] = vstage[p];
        }
    }
}

// Up to RS_SMALL keys (RS_SMALL_KV with values) are sorted by one workgroup in one
// launch: keys in registers, LDS between the passes.  The batches of an edge stream
// are this short, and three launches of 5 to 8 us (gaps included) per eight bits
// bounded them: 2,000 keys of 32 bits 97 us, 11.5 so; one CU ranks 8,192 keys of 49
// bits in 23 us.
constexpr int RS_SMALL_BLOCK = 1024;
constexpr int64_t RS_SMALL = RS_SMALL_BLOCK * 16, RS_SMALL_KV = RS_SMALL_BLOCK * 8;   // what 160 KB of LDS hold

// what it sorts: keys (and values) in place, or pairs, packed as they are loaded
struct SmallKeys {
    const uint64_t* k;
    const uint32_t* v;
    __device__ __forceinline__ void begin() const {}
    __device__ __forceinline__ uint64_t key(int i) const { return k[i]; }
    __device__ __forceinline__ uint32_t val(int i) const { return v[i]; }
};
struct SmallPairs {
    SortPairs p;
    __device__ __forceinline__ void begin() const {
        if ((int)threadIdx.x < p.words) p.state[threadIdx.x] = 0;
        __syncthreads();   // before any error is noted
    }
    __device__ __forceinline__ uint64_t key(int i) const {
        const int32_t s = p.src[i], d = p.dst[i];
        if (s < 0 || s >= p.nv || d < 0 || d >= p.nv) {
            atomicOr(p.err, p.bad);
            return 0;
        }
        return ((uint64_t)s << p.sbits) | (uint64_t)d;
    }
    __device__ __forceinline__ uint32_t val(int i) const { return (uint32_t)i; }
};

template <bool KV, int IPT, typename Src>
__global__ __launch_bounds__(RS_SMALL_BLOCK) void rs_small_kernel(Src in, uint64_t* keys, uint32_t* vals, int n,
                                                                  int key_bits) {
    constexpr int WAVES = RS_SMALL_BLOCK / WAVE;
    __shared__ uint64_t stage[RS_SMALL_BLOCK * IPT];
    __shared__ uint32_t vstage[KV ? RS_SMALL_BLOCK * IPT : 1];
    __shared__ uint32_t cnt[WAVES][RS_BUCKETS];   // a wave's digit counts, then the starts of its keys
    __shared__ uint32_t wtot[RS_BUCKETS / WAVE];
    const int w = threadIdx.x / WAVE;
    const int l = __lane_id();
    const int rows = (n + RS_SMALL_BLOCK - 1) / RS_SMALL_BLOCK;
    const int base = w * rows * WAVE;
    const uint64_t lt = lanemask_lt();
    in.begin();
    // past the end: the largest key, which a stable sort leaves there
    uint64_t k[IPT];
    uint32_t v[IPT], rank[IPT];
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const int i = base + j * WAVE + l;
        const bool any = j < rows && i < n;
        k[j] = any ? in.key(i) : ~0ull;
        v[j] = KV && any ? in.val(i) : 0u;
    }
    for (int shift = 0; shift < key_bits; shift += RS_BITS) {
        for (int d = threadIdx.x; d < WAVES * RS_BUCKETS; d += RS_SMALL_BLOCK) (&cnt[0][0])[d] = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IPT; j++) {
            if (j >= rows) continue;
            const uint32_t d = (uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1);
            uint64_t peers = ~0ull;
#pragma unroll
            for (int b = 0; b < RS_BITS; b++) {
                const uint64_t bal = __ballot((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? bal : ~bal;
            }
            const uint32_t before = (uint32_t)__popcll(peers & lt);
            const uint32_t start = cnt[w][d];
            rank[j] = start + before;
            // the lowest peer lane publishes the new count after every peer has read it
            if (before == 0) cnt[w][d] = start + (uint32_t)__popcll(peers);
        }
        __syncthreads();
        uint32_t run = 0, inc = 0;
        if (threadIdx.x < RS_BUCKETS) {
#pragma unroll
            for (int q = 0; q < WAVES; q++) run += cnt[q][threadIdx.x];
            inc = wave_inclusive_scan(run);
            if (l == WAVE - 1) wtot[w] = inc;
        }
        __syncthreads();
        if (threadIdx.x < RS_BUCKETS) {
            uint32_t at = inc - run;
            for (int q = 0; q < w; q++) at += wtot[q];
#pragma unroll
            for (int q = 0; q < WAVES; q++) {
                const uint32_t c = cnt[q][threadIdx.x];
                cnt[q][threadIdx.x] = at;
                at += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IPT; j++) {
            if (j >= rows) continue;
            const uint32_t p = cnt[w][(uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1)] + rank[j];
            stage[p] = k[j];
            if constexpr (KV) vstage[p] = v[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IPT; j++) {
            if (j >= rows) continue;
            k[j] = stage[base + j * WAVE + l];
            if constexpr (KV) v[j] = vstage[base + j * WAVE + l];
        }
    }
#pragma unroll
    for (int j = 0; j < IPT; j++) {
        const int i = base + j * WAVE + l;
        if (j < rows && i < n) {
            keys[i] = k[j];
            if constexpr (KV) vals[i] = v[j];
        }
    }
}

}  // namespace

// Resolves this file's code object (see preload_code_objects in graph.hip).
void preload_prims_code() {
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&rs_rowscan_kernel)) != hipSuccess) (void)hipGetLastError();
}

// Keys per tile: few where tiles are few, as a pass is then one tile's chain (100 K
// keys, per pass: 10.6 us with 1,024, 12.5 with 2,048, 16.5 with 4,096; 2 M keys:
// 27, 24 and 26); many where they are many, as runs are then longer and there are
// fewer counts (67 M keys: 690, 484 and 393; 8,192 in workgroups of 512 lanes: 403).
constexpr int64_t RS_FINE = (int64_t)1 << 20, RS_MIDDLE = (int64_t)1 << 23;
static int64_t rs_tile_keys(int64_t n) { return n < RS_FINE ? 256 * 4 : n < RS_MIDDLE ? 256 * 8 : 256 * 16; }

// tiles of the largest sort of up to n keys (fewer keys may take more of them)
static int64_t rs_max_tiles(int64_t n) {
    int64_t t = ceil_div(n, rs_tile_keys(n));
    for (const int64_t edge : {RS_FINE - 1, RS_MIDDLE - 1})
        if (n > edge) t = std::max(t, ceil_div(edge, rs_tile_keys(edge)));
    return t;
}

size_t sort_temp_bytes(int64_t n) {
    const int64_t hn_ = rs_max_tiles(n > 0 ? n : 1) * RS_BUCKETS;
    return (size_t)(hn_ + 1) * 4 * 2 + RS_BUCKETS * 4 + 512;
}

template <int THREADS, int IPT>
static hn_status rs_pass(const uint64_t* in, uint64_t* out, const uint32_t* vin, uint32_t* vout, int64_t n, int shift,
                         uint32_t* hist, uint32_t* hoff, uint32_t* dtot, hipStream_t st) {
    const int64_t tiles = ceil_div(n, THREADS * IPT);
    rs_hist_kernel<THREADS, IPT><<<(unsigned)tiles, THREADS, 0, st>>>(in, n, shift, tiles, hist);
    HN_CHECK_LAUNCH();
    rs_rowscan_kernel<<<RS_BUCKETS, BLOCK, 0, st>>>(hist, tiles, hoff, dtot);
    HN_CHECK_LAUNCH();
    if (vin)
        rs_scatter_kernel<true, THREADS, IPT><<<(unsigned)tiles, THREADS, 0, st>>>(in, n, shift, tiles, hoff, dtot, out,
                                                                                   vin, vout);
    else
        rs_scatter_kernel<false, THREADS, IPT><<<(unsigned)tiles, THREADS, 0, st>>>(in, n, shift, tiles, hoff, dtot,
                                                                                    out, nullptr, nullptr);
    HN_CHECK_LAUNCH();
    return HN_OK;
}

int64_t sort_small_max(bool values) { return values ? RS_SMALL_KV : RS_SMALL; }

template <typename Src>
static hn_status rs_small(Src in, uint64_t* keys, uint32_t* vals, int64_t n, int key_bits, hipStream_t st) {
    if (vals) rs_small_kernel<true, 8><<<1, RS_SMALL_BLOCK, 0, st>>>(in, keys, vals, (int)n, key_bits);
    else if (n <= RS_SMALL_BLOCK * 8) rs_small_kernel<false, 8><<<1, RS_SMALL_BLOCK, 0, st>>>(in, keys, vals, (int)n, key_bits);
    else rs_small_kernel<false, 16><<<1, RS_SMALL_BLOCK, 0, st>>>(in, keys, vals, (int)n, key_bits);
    HN_CHECK_LAUNCH();
    return HN_OK;
}

hn_status radix_sort_small_pairs(const SortPairs& pairs, uint64_t* keys, uint32_t* idx, int64_t n, int key_bits,
                                 hipStream_t st) {
    return rs_small(SmallPairs{pairs}, keys, idx, n, key_bits, st);
}

static hn_status radix_sort_impl(uint64_t** keys, uint64_t** alt, uint32_t** vals, uint32_t** valt, int64_t n,
                                 int key_bits, void* tmp, hipStream_t st) {
    if (n <= 1) return HN_OK;
    if (n <= sort_small_max(vals != nullptr))
        return rs_small(SmallKeys{*keys, vals ? *vals : nullptr}, *keys, vals ? *vals : nullptr, n, key_bits, st);
    const int64_t tile = rs_tile_keys(n);
    const int64_t hn_ = ceil_div(n, tile) * RS_BUCKETS;
    HN_ARG(hn_ < (int64_t)0xFFFFFFFF && n < (int64_t)0xFFFFFFFF, "radix_sort_u64: too many keys");
    uint32_t* hist = reinterpret_cast<uint32_t*>(tmp);
    uint32_t* hoff = hist + hn_ + 1;
    uint32_t* dtot = hoff + hn_ + 1;   // RS_BUCKETS digit totals
    for (int shift = 0; shift < key_bits; shift += RS_BITS) {
        const uint32_t* vin = vals ? *vals : nullptr;
        uint32_t* vout = vals ? *valt : nullptr;
        if (tile == 256 * 4) HN_TRY((rs_pass<256, 4>(*keys, *alt, vin, vout, n, shift, hist, hoff, dtot, st)));
        else if (tile == 256 * 8) HN_TRY((rs_pass<256, 8>(*keys, *alt, vin, vout, n, shift, hist, hoff, dtot, st)));
        else HN_TRY((rs_pass<256, 16>(*keys, *alt, vin, vout, n, shift, hist, hoff, dtot, st)));
        std::swap(*keys, *alt);
        if (vals) std::swap(*vals, *valt);
    }
    return HN_OK;
}

hn_status radix_sort_u64(uint64_t** keys, uint64_t** alt, int64_t n, int key_bits, void* tmp, hipStream_t st) {
    return radix_sort_impl(keys, alt, nullptr, nullptr, n, key_bits, tmp, st);
}

hn_status radix_sort_u64_kv(uint64_t** keys, uint64_t** alt, uint32_t** vals, uint32_t** valt, int64_t n,
                            int key_bits, void* tmp, hipStream_t st) {
    return radix_sort_impl(keys, alt, vals, valt, n, key_bits, tmp, st);
}

}  // namespace hn
