// Compile-time sorting and merging networks over a lane's registers (every
// index is a constant, so the arrays stay in registers).
#pragma once

#include "common.h"

#ifdef __HIPCC__
namespace tgn {

// Knuth's merge exchange (The Art of Computer Programming 3, 5.2.2 M) for any
// N: for p = 2^(t-1) .. 1, compare (i, i + p) where i & p == 0, then
// (i, i + q - p) where i & p for q = 2^(t-1) .. 2p.
template <int D, int P, int R, int N, typename K>
__device__ __forceinline__ void sort_stage(K (&k)[N]) {
#pragma unroll
    for (int i = 0; i < N - D; i++)
        if ((i & P) == R) {
            const K a = k[i], b = k[i + D];
            k[i] = tgd::opaque(min(a, b));
            k[i + D] = tgd::opaque(max(a, b));
        }
}
template <int P, int Q, int N, typename K>
__device__ __forceinline__ void sort_merges(K (&k)[N]) {
    if constexpr (Q > P) {
        sort_stage<Q - P, P, P>(k);
        sort_merges<P, Q / 2>(k);
    }
}
template <int P, int TOP, int N, typename K>
__device__ __forceinline__ void sort_phases(K (&k)[N]) {
    if constexpr (P > 0) {
        sort_stage<P, P, 0>(k);
        sort_merges<P, TOP>(k);
        sort_phases<P / 2, TOP>(k);
    }
}
constexpr int top_power(int n) { return n <= 2 ? 1 : 2 * top_power((n + 1) / 2); }  // 2^(ceil(log2 n) - 1)
template <int N, typename K>
__device__ __forceinline__ void sort_keys(K (&k)[N]) {
    sort_phases<top_power(N), top_power(N)>(k);
}

// Bitonic merge of k[B .. B + n), any n: the first part sorted against the
// direction, the second along it (H. W. Lang's form for arbitrary n: compare
// at the largest power of two below n, then both parts).
constexpr int pow2_below(int n) { return n <= 2 ? 1 : 2 * pow2_below((n + 1) / 2); }
template <int B, int n, bool UP, int N>
__device__ __forceinline__ void bitonic_merge(int32_t (&k)[N]) {
    if constexpr (n > 1) {
        constexpr int m = pow2_below(n);
#pragma unroll
        for (int i = B; i < B + n - m; i++) {
            const int32_t a = k[i], b = k[i + m];
            k[i] = tgd::opaque(UP ? min(a, b) : max(a, b));
            k[i + m] = tgd::opaque(UP ? max(a, b) : min(a, b));
        }
        bitonic_merge<B, m, UP>(k);
        bitonic_merge<B + m, n - m, UP>(k);
    }
}

}  // namespace tgn
#endif
