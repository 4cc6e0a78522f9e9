// Sorted column sets in LDS, one per thread: the rows of a sparsity pattern
// while it is built (element patterns, Galerkin coarse operators).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

// Per-thread sorted column set in LDS (layout set[k*B + tid]).
template <int B>
__device__ __forceinline__ bool set_insert(int32_t *set, int &n, int rmax, int32_t c)
{
    const int t = threadIdx.x;
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        int32_t v = set[mid * B + t];
        if (v < c) lo = mid + 1;
        else hi = mid;
    }
    if (lo < n && set[lo * B + t] == c) return true;
    if (n >= rmax) return false;
    for (int k = n; k > lo; --k) set[k * B + t] = set[(k - 1) * B + t];
    set[lo * B + t] = c;
    ++n;
    return true;
}

template <int B>
__device__ __forceinline__ int set_find(const int32_t *set, int n, int32_t c)
{
    const int t = threadIdx.x;
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (set[mid * B + t] < c) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}
