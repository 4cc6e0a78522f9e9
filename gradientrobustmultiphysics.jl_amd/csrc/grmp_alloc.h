// Allocation with one retry: out of memory, what can be released is released
// first and the allocation tried again.
#pragma once
#include <hip/hip_runtime_api.h>

template <class Alloc, class Release>
inline hipError_t alloc_or_release(Alloc alloc, Release release)
{
    const hipError_t e = alloc();
    if (e != hipErrorOutOfMemory) return e;
    release();
    return alloc();
}
