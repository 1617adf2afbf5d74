// hostcopy.h -- device arrays to the caller's pageable host arrays (hostcopy.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <mutex>
#include <vector>

namespace pictor {

// One array to deliver: `n` elements of `elem` bytes at dst, from device memory.  kind: kRaw copies;
// the others make FP64 of a split-form array (kPair: src + lo; kFloat: src; kScaled: scale * FP64 src).
struct HostItem {
    enum Kind { kRaw, kPair, kFloat, kScaled } kind = kRaw;
    void *dst = nullptr;
    const void *src = nullptr;
    const float *lo = nullptr;
    double scale = 1.0;
    size_t n = 0, elem = 8;
};

// The pinned ring behind deliver(), one per context: at most 32 MiB, given back with it; one call
// at a time uses it (lock).
struct HostRing {
    std::mutex lock;
    char *buf = nullptr;
    int slots = 0;
    std::vector<hipEvent_t> ev;
    void release();
};

// One array as it is.
inline HostItem host_raw(void *dst, const void *src, size_t n, size_t elem)
{
    HostItem it;
    it.dst = dst;
    it.src = src;
    it.n = n;
    it.elem = elem;
    return it;
}

// Copies every item to its host array; returns when all have arrived.  hipSuccess or the first error.
hipError_t deliver(HostRing &ring, const std::vector<HostItem> &items, hipStream_t s);

}  // namespace pictor
