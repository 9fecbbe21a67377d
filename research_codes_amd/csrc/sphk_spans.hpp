// sphk_spans.hpp -- which cells a particle of a sorted key array begins: the
// parts of the tree build that need no GPU (host and device).
#ifndef SPHK_SPANS_HPP
#define SPHK_SPANS_HPP

#include <cstdint>

#ifdef __HIPCC__
#define SPHK_HD __host__ __device__ __forceinline__
#else
#define SPHK_HD inline
#endif

namespace sphk {

constexpr int kMaxLevel = 21;   // 21 bits per dimension, three to a digit

// Leading digits that two keys share.
SPHK_HD int shared_digits(uint64_t a, uint64_t b)
{
    return a == b ? kMaxLevel : (__builtin_clzll(a ^ b) - 1) / 3;
}

// Deepest level at which the cell of particle i holds more than n_leaf of the
// n particles (-1: none).  Cells nest, so the level is bisected; a cell holds
// more than n_leaf if its first particle and the one n_leaf places on are both
// in it, and the first that matters lies at most n_leaf places before i.  At
// most 5 (log2(n_leaf) + 3) keys are read, where the windows of n_leaf + 1
// particles around i would take 2 (n_leaf + 1).  Keys out of order give some
// level; the build refuses them.
template <class Keys>
SPHK_HD int deepest_full_level(const Keys &key, int n, int n_leaf, int i)
{
    if (n <= n_leaf) return -1;
    const uint64_t own = key[i];
    const int first = i > n_leaf ? i - n_leaf : 0;
    int lo = 0, hi = kMaxLevel;   // full at lo (the root's cell is), not beyond hi
    while (lo < hi) {
        const int L = (lo + hi + 1) / 2, shift = 3 * (kMaxLevel - L);
        const uint64_t p = own >> shift;
        int b = first, e = i;     // the first of [first, i] that is in the cell
        while (b < e) {
            const int mid = b + (e - b) / 2;
            if (key[mid] >> shift == p)
                e = mid;
            else
                b = mid + 1;
        }
        if (b < n - n_leaf && key[b + n_leaf] >> shift == p)
            lo = L;
        else
            hi = L - 1;
    }
    return lo;
}

}  // namespace sphk

#endif
