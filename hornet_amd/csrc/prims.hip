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

#include <utility>

namespace hn {

// ------------------------------------------------------------------ radix sort
namespace {

constexpr int RS_BITS = 8;
constexpr int RS_BUCKETS = 1 << RS_BITS;
constexpr int RS_IPT = 16;                      // keys per lane
constexpr int RS_TILE = BLOCK * RS_IPT;         // 4096 keys
constexpr int RS_WAVE_KEYS = WAVE * RS_IPT;     // 1024 keys per wave
static_assert(RS_BUCKETS == BLOCK, "one thread per digit in the per-digit steps");

__global__ __launch_bounds__(BLOCK) void rs_hist_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                        int shift, int64_t ntiles,
                                                        uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[RS_BUCKETS];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * RS_TILE;
#pragma unroll 4
    for (int j = 0; j < RS_IPT; j++) {
        int64_t i = base + (int64_t)j * BLOCK + threadIdx.x;
        if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & (RS_BUCKETS - 1)], 1u);
    }
    __syncthreads();
    hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = cnt[threadIdx.x];
}

// Per digit (one workgroup each): exclusive prefix of its per-tile counts
// across the tiles, and the digit's total.  The scatter adds the digit's start
// (prefix of the totals over smaller digits), so a pass needs no global scan.
__global__ __launch_bounds__(BLOCK) void rs_rowscan_kernel(const uint32_t* __restrict__ hist, int64_t ntiles,
                                                           uint32_t* __restrict__ hoff, uint32_t* __restrict__ dtot) {
    __shared__ uint32_t sc[NWAVES + 1];
    const uint32_t* row = hist + (int64_t)blockIdx.x * ntiles;
    uint32_t* out = hoff + (int64_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (int64_t t0 = 0; t0 < ntiles; t0 += BLOCK) {
        const int64_t t = t0 + threadIdx.x;
        const uint32_t x = t < ntiles ? row[t] : 0u;
        uint32_t tot;
        const uint32_t ex = block_exclusive_scan(x, sc, &tot);
        if (t < ntiles) out[t] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) dtot[blockIdx.x] = carry;
}

// KV: a 32-bit value rides with each key (staged beside it in LDS)
template <bool KV>
__global__ __launch_bounds__(BLOCK) void rs_scatter_kernel(const uint64_t* __restrict__ keys, int64_t n,
                                                           int shift, int64_t ntiles,
                                                           const uint32_t* __restrict__ hoff,
                                                           const uint32_t* __restrict__ dtot,
                                                           uint64_t* __restrict__ out,
                                                           const uint32_t* __restrict__ vin,
                                                           uint32_t* __restrict__ vout) {
    __shared__ uint32_t wcnt[NWAVES][RS_BUCKETS];   // per-wave digit counts
    __shared__ uint32_t dstart[RS_BUCKETS];         // tile-local start of each digit
    __shared__ uint32_t gbase[RS_BUCKETS];          // global start of this tile's digit run
    __shared__ uint64_t stage[RS_TILE];
    __shared__ uint32_t vstage[KV ? RS_TILE : 1];
    __shared__ uint32_t sc[NWAVES + 1];

    const int w = threadIdx.x / WAVE;
    const int l = __lane_id();
    for (int d = threadIdx.x; d < NWAVES * RS_BUCKETS; d += BLOCK) (&wcnt[0][0])[d] = 0;
    __syncthreads();

    const int64_t base = (int64_t)blockIdx.x * RS_TILE + (int64_t)w * RS_WAVE_KEYS;
    uint64_t k[RS_IPT];
    uint32_t rank[RS_IPT];
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int j = 0; j < RS_IPT; j++) {
        int64_t i = base + (int64_t)j * WAVE + l;
        bool valid = i < n;
        k[j] = valid ? keys[i] : 0;
        uint32_t d = (uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1);
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < RS_BITS; b++) {
            uint64_t bal = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? bal : ~bal;
        }
        uint32_t before = (uint32_t)__popcll(peers & lt);
        uint32_t cntp = (uint32_t)__popcll(peers);
        uint32_t basec = valid ? wcnt[w][d] : 0;
        rank[j] = basec + before;
        // the lowest peer lane publishes the new count after every peer has read it
        if (valid && before == 0) wcnt[w][d] = basec + cntp;
    }
    __syncthreads();
    // per digit: totals over waves, exclusive across waves
    {
        const int d = threadIdx.x;
        uint32_t run = 0;
#pragma unroll
        for (int q = 0; q < NWAVES; q++) {
            uint32_t c = wcnt[q][d];
            wcnt[q][d] = run;
            run += c;
        }
        uint32_t tot;
        uint32_t ex = block_exclusive_scan(run, sc, &tot);
        dstart[d] = ex;
        // digit d starts after every key of the smaller digits
        const uint32_t dbase = block_exclusive_scan(dtot[d], sc, &tot);
        gbase[d] = dbase + hoff[(int64_t)d * ntiles + blockIdx.x];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RS_IPT; j++) {
        int64_t i = base + (int64_t)j * WAVE + l;
        if (i < n) {
            uint32_t d = (uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1);
            stage[dstart[d] + wcnt[w][d] + rank[j]] = k[j];
            if constexpr (KV) vstage[dstart[d] + wcnt[w][d] + rank[j]] = vin[i];
        }
    }
    __syncthreads();
    const int64_t tile_n = min((int64_t)RS_TILE, n - (int64_t)blockIdx.x * RS_TILE);
    for (int p = threadIdx.x; p < tile_n; p += BLOCK) {
        uint64_t key = stage[p];
        uint32_t d = (uint32_t)(key >> shift) & (RS_BUCKETS - 1);
        out[(int64_t)gbase[d] + (p - dstart[d])] = key;
        if constexpr (KV) vout[(int64_t)gbase[d] + (p - dstart[d])] = vstage[p];
    }
}

// Up to RS_SMALL keys are sorted by one workgroup in one launch: keys in registers,
// LDS between the passes.  The batches of an edge stream are this short, and three
// launches of 8 us (gaps included) per eight bits bounded them: 2,000 keys of 32 bits
// 97 us, 11.5 so.  One CU ranks 8,192 keys of 49 bits in 23 us, about what the
// launches' kernels alone take for as many; beyond that the whole device is faster.
constexpr int RS_SMALL_BLOCK = 1024;
constexpr int RS_SMALL_IPT = 8;
constexpr int RS_SMALL = RS_SMALL_BLOCK * RS_SMALL_IPT;

template <bool KV>
__global__ __launch_bounds__(RS_SMALL_BLOCK) void rs_small_kernel(uint64_t* __restrict__ keys,
                                                                  uint32_t* __restrict__ vals, int n, int key_bits) {
    constexpr int WAVES = RS_SMALL_BLOCK / WAVE;
    __shared__ uint64_t stage[RS_SMALL];
    __shared__ uint32_t vstage[KV ? RS_SMALL : 1];
    __shared__ uint32_t cnt[WAVES][RS_BUCKETS];   // a wave's digit counts, then the starts of its keys
    __shared__ uint32_t wtot[RS_BUCKETS / WAVE];
    const int w = threadIdx.x / WAVE;
    const int l = __lane_id();
    const int rows = (n + RS_SMALL_BLOCK - 1) / RS_SMALL_BLOCK;
    const int base = w * rows * WAVE;
    const uint64_t lt = lanemask_lt();
    // past the end: the largest key, which a stable sort leaves there
    uint64_t k[RS_SMALL_IPT];
    uint32_t v[RS_SMALL_IPT], rank[RS_SMALL_IPT];
#pragma unroll
    for (int j = 0; j < RS_SMALL_IPT; j++) {
        const int i = base + j * WAVE + l;
        const bool in = j < rows && i < n;
        k[j] = in ? keys[i] : ~0ull;
        v[j] = KV && in ? vals[i] : 0u;
    }
    for (int shift = 0; shift < key_bits; shift += RS_BITS) {
        for (int d = threadIdx.x; d < WAVES * RS_BUCKETS; d += RS_SMALL_BLOCK) (&cnt[0][0])[d] = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < RS_SMALL_IPT; j++) {
            if (j >= rows) break;
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
        for (int j = 0; j < RS_SMALL_IPT; j++) {
            if (j >= rows) break;
            const uint32_t p = cnt[w][(uint32_t)(k[j] >> shift) & (RS_BUCKETS - 1)] + rank[j];
            stage[p] = k[j];
            if constexpr (KV) vstage[p] = v[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < RS_SMALL_IPT; j++) {
            if (j >= rows) break;
            k[j] = stage[base + j * WAVE + l];
            if constexpr (KV) v[j] = vstage[base + j * WAVE + l];
        }
    }
#pragma unroll
    for (int j = 0; j < RS_SMALL_IPT; j++) {
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
    if (hipFuncGetAttributes(&a, reinterpret_cast<const void*>(&rs_hist_kernel)) != hipSuccess) (void)hipGetLastError();
}

size_t sort_temp_bytes(int64_t n) {
    int64_t tiles = ceil_div(n > 0 ? n : 1, RS_TILE);
    int64_t hn_ = tiles * RS_BUCKETS;
    return (size_t)(hn_ + 1) * 4 * 2 + scan_temp_bytes(hn_) + RS_BUCKETS * 4 + 512;
}

static hn_status radix_sort_impl(uint64_t** keys, uint64_t** alt, uint32_t** vals, uint32_t** valt, int64_t n,
                                 int key_bits, void* tmp, hipStream_t st) {
    if (n <= 1) return HN_OK;
    if (n <= RS_SMALL) {
        if (vals) rs_small_kernel<true><<<1, RS_SMALL_BLOCK, 0, st>>>(*keys, *vals, (int)n, key_bits);
        else rs_small_kernel<false><<<1, RS_SMALL_BLOCK, 0, st>>>(*keys, nullptr, (int)n, key_bits);
        HN_CHECK_LAUNCH();
        return HN_OK;
    }
    int64_t tiles = ceil_div(n, RS_TILE);
    int64_t hn_ = tiles * RS_BUCKETS;
    HN_ARG(hn_ < (int64_t)0xFFFFFFFF && n < (int64_t)0xFFFFFFFF, "radix_sort_u64: too many keys");
    uint32_t* hist = reinterpret_cast<uint32_t*>(tmp);
    uint32_t* hoff = hist + hn_ + 1;
    void* stmp = reinterpret_cast<char*>(tmp) + (size_t)(hn_ + 1) * 4 * 2 + 256;
    stmp = reinterpret_cast<void*>((reinterpret_cast<uintptr_t>(stmp) + 255) & ~uintptr_t(255));
    uint32_t* dtot = reinterpret_cast<uint32_t*>(stmp);   // RS_BUCKETS digit totals
    for (int shift = 0; shift < key_bits; shift += RS_BITS) {
        rs_hist_kernel<<<(unsigned)tiles, BLOCK, 0, st>>>(*keys, n, shift, tiles, hist);
        HN_CHECK_LAUNCH();
        rs_rowscan_kernel<<<RS_BUCKETS, BLOCK, 0, st>>>(hist, tiles, hoff, dtot);
        HN_CHECK_LAUNCH();
        if (vals)
            rs_scatter_kernel<true><<<(unsigned)tiles, BLOCK, 0, st>>>(*keys, n, shift, tiles, hoff, dtot, *alt,
                                                                       *vals, *valt);
        else
            rs_scatter_kernel<false><<<(unsigned)tiles, BLOCK, 0, st>>>(*keys, n, shift, tiles, hoff, dtot, *alt,
                                                                        nullptr, nullptr);
        HN_CHECK_LAUNCH();
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
