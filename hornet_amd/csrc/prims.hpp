// prims.hpp -- status-returning wrappers of the shared wave64 scan
// (include/hornet/detail/wave.hpp) for the library.
#pragma once
#include "common.hpp"

namespace hn {

inline hn_status scan_status(hipError_t e) {
    if (e == hipSuccess) return HN_OK;
    set_error(std::string("scan launch: ") + hipGetErrorString(e));
    return HN_E_HIP;
}

// Exclusive scan of in(0..n) delivered to out(i, prefix, value); *total = sum.
template <typename Out, typename InFn, typename OutFn>
hn_status exclusive_scan_fn(InFn in, OutFn out, Out* total, int64_t n, void* tmp, hipStream_t st) {
    return scan_status(exclusive_scan_dev<Out>(in, out, total, n, tmp, st));
}

template <typename Out, typename InFn, typename OutFn>
ScanOf<Out, InFn, OutFn> scan_of(InFn in, OutFn out, Out* total, int64_t n) {
    return {in, out, total, n};
}

// Scan a, then scan b, which may read what a wrote: one launch where both are of at
// most SCAN_ONE values, otherwise two scans.
template <typename A, typename B>
hn_status exclusive_scan_two(const A& a, const B& b, void* tmp, hipStream_t st) {
    if (a.n > 0 && b.n > 0 && a.n <= SCAN_ONE && b.n <= SCAN_ONE) {
        scan_two_kernel<A, B><<<1, SCAN_ONE_BLOCK, 0, st>>>(a, b);
        return scan_status(hipGetLastError());
    }
    const hn_status s = exclusive_scan_fn<typename A::Out>(a.in, a.out, a.total, a.n, tmp, st);
    return s != HN_OK ? s : exclusive_scan_fn<typename B::Out>(b.in, b.out, b.total, b.n, tmp, st);
}

// out[0..n) = exclusive prefix of in(0..n), out[n] = total.
template <typename Out, typename InFn>
hn_status exclusive_scan(InFn in, Out* out, int64_t n, void* tmp, hipStream_t st) {
    return scan_status(exclusive_scan_dev<Out>(in, ArrayOut<Out>{out}, out + n, n, tmp, st));
}

}  // namespace hn
