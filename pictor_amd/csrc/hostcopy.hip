// hostcopy.hip -- results to pageable host memory.
//
// A copy into freshly allocated host memory is bound by the host: the runtime's own path (a device
// copy into its staging buffer, one thread copying out and taking the page faults) delivers 303 MB
// (2048 x 2048, nine FP64 arrays) in 31.7 ms, 76 MB in 8.7 ms and 0.3 MB in 0.32 ms.  Here kernels
// write into a ring of pinned 1 MiB chunks (the split form's fields become FP64 on the way, without
// a device copy) and host threads copy chunks out while later ones arrive, faulting pages in
// parallel: 8.1, 2.2 and 0.08 ms.  The kernel write matters: a piece sent by hipMemcpyAsync costs
// 20 us of launch, and the 303 MB take 11.2 ms.  Small arrays share a chunk and its wait, and the
// caller alone copies results of up to kThreadBytes: starting threads would take longer.
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>

namespace pictor {
namespace {

// piece size: 0.25 MiB pieces deliver the 303 MB in 12.0 ms, 0.5 MiB in 9.1, 1 MiB in 8.1, 2 MiB in 7.5
constexpr size_t kChunk = 1 << 20;
// chunks in the ring: at most 32 MiB of pinned memory, and a share of the result, since pinning
// costs 0.4 ms per MiB in a context's first download
constexpr size_t kSlots = 32;
constexpr size_t kSlotShare = 3 << 20;
constexpr size_t kSlotsAlone = 2;
constexpr int kThreads = 8;                // one per kThreadShare bytes, at most this many
constexpr size_t kThreadShare = 3 << 20;
constexpr size_t kThreadBytes = 6 << 20;   // 4.9 MB: alone 0.46 ms, 8 threads 0.55; 9.6 MB: 3 threads 0.77 ms

__global__ __launch_bounds__(256) void k_to_host(int kind, const void *__restrict__ src, const float *__restrict__ lo,
                                                 double scale, size_t off, int n, double *__restrict__ out)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const size_t i = off + t;
    if (kind == HostItem::kPair) out[t] = (double)((const float *)src)[i] + (double)lo[i];
    else if (kind == HostItem::kFloat) out[t] = (double)((const float *)src)[i];
    else out[t] = ((const double *)src)[i] * scale;
}

// n 4-byte words, both sides on 16-byte boundaries
__global__ __launch_bounds__(256) void k_words_to_host(const uint4 *__restrict__ src, int n, uint4 *__restrict__ out)
{
    const int t = blockIdx.x * 256 + threadIdx.x, r = n - 4 * t;
    if (r >= 4) out[t] = src[t];
    else if (r > 0)
        for (int j = 0; j < r; j++) ((unsigned *)(out + t))[j] = ((const unsigned *)(src + t))[j];
}

// elements off .. off + n - 1 of an item, at byte `at` of its batch
struct Piece {
    const HostItem *item;
    size_t off, n, at;
    size_t bytes() const { return n * item->elem; }
    char *dst() const { return (char *)item->dst + off * item->elem; }
};

// pieces first .. last - 1 fill one chunk of the ring
struct Batch {
    size_t first, last;
};

// piece p to `to`: memory that the device can write (by_kernel), or any host memory (kRaw only)
hipError_t enqueue(const Piece &p, char *to, hipStream_t s, bool by_kernel = true)
{
    const HostItem &it = *p.item;
    if (it.kind == HostItem::kRaw) {
        const char *src = (const char *)it.src + p.off * it.elem;
        if (!by_kernel || (uintptr_t)src % 16 || p.bytes() % 4)
            return hipMemcpyAsync(to, src, p.bytes(), hipMemcpyDeviceToHost, s);
        const int words = (int)(p.bytes() / 4);
        hipLaunchKernelGGL(k_words_to_host, dim3((words + 1023) / 1024), dim3(256), 0, s, (const uint4 *)src, words,
                           (uint4 *)to);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_to_host, dim3((unsigned)((p.n + 255) / 256)), dim3(256), 0, s, (int)it.kind, it.src, it.lo,
                       it.scale, p.off, (int)p.n, (double *)to);
    return hipGetLastError();
}

// the ring with `want` chunks, 1 <= want <= kSlots; false: no pinned memory or events
bool grow(HostRing &r, int want)
{
    while ((int)r.ev.size() < want) {
        hipEvent_t v;
        if (hipEventCreateWithFlags(&v, hipEventDisableTiming) != hipSuccess) return false;
        r.ev.push_back(v);
    }
    if (r.slots >= want) return true;
    if (r.buf) (void)hipHostFree(r.buf);
    r.buf = nullptr;
    r.slots = 0;
    if (hipHostMalloc((void **)&r.buf, kChunk * want, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        r.buf = nullptr;
        return false;
    }
    r.slots = want;
    return true;
}

// an array in memory that the device reaches (the caller's pinned or managed memory): straight into it
hipError_t deliver_mapped(const HostItem &it, hipStream_t s, bool &done)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, it.dst) != hipSuccess) {
        (void)hipGetLastError();
        return hipSuccess;
    }
    if (a.type == hipMemoryTypeUnregistered || !a.devicePointer) return hipSuccess;
    done = true;
    if (it.kind == HostItem::kRaw) return hipMemcpyAsync(it.dst, it.src, it.n * it.elem, hipMemcpyDefault, s);
    constexpr size_t per = 1 << 26;   // elements of a launch
    for (size_t o = 0; o < it.n; o += per) {
        const Piece p{&it, o, std::min(per, it.n - o), 0};
        const hipError_t e = enqueue(p, (char *)a.devicePointer + o * it.elem, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// without pinned memory: the runtime's own copies, converted pieces through a device chunk
hipError_t deliver_plain(const std::vector<Piece> &todo, hipStream_t s)
{
    hipError_t e = hipSuccess;
    char *chunk = nullptr;
    for (const Piece &p : todo) {
        if (p.item->kind == HostItem::kRaw) {
            e = enqueue(p, p.dst(), s, false);
        } else {
            if (!chunk) e = hipMalloc((void **)&chunk, kChunk);
            if (e == hipSuccess) e = enqueue(p, chunk, s);
            if (e == hipSuccess) e = hipMemcpyAsync(p.dst(), chunk, p.bytes(), hipMemcpyDeviceToHost, s);
        }
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e != hipSuccess) break;
    }
    if (chunk) (void)hipFree(chunk);
    return e;
}

}  // namespace

void HostRing::release()
{
    if (buf) (void)hipHostFree(buf);
    for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    buf = nullptr;
    slots = 0;
    ev.clear();
}

hipError_t deliver(HostRing &ring, const std::vector<HostItem> &items, hipStream_t s)
{
    std::lock_guard<std::mutex> own(ring.lock);
    std::vector<Piece> todo;
    std::vector<Batch> batch;
    size_t bytes = 0, used = kChunk;   // of the last batch
    for (const HostItem &it : items) {
        bool direct = false;
        const hipError_t d = deliver_mapped(it, s, direct);
        if (d != hipSuccess) return d;
        if (direct) continue;
        const size_t per = kChunk / it.elem;
        for (size_t o = 0; o < it.n; o += per) {
            Piece p{&it, o, std::min(per, it.n - o), 0};
            if (used + p.bytes() > kChunk) {
                batch.push_back({todo.size(), todo.size()});
                used = 0;
            }
            p.at = used;
            used += (p.bytes() + 63) / 64 * 64;
            batch.back().last++;
            todo.push_back(p);
        }
        bytes += it.n * it.elem;
    }
    if (todo.empty()) return hipStreamSynchronize(s);
    const size_t nb = batch.size();
    const bool alone = bytes <= kThreadBytes;
    const size_t slots = std::min(nb, alone ? kSlotsAlone : std::min(kSlots, bytes / kSlotShare));
    if (!grow(ring, (int)slots)) return deliver_plain(todo, s);

    // batch k goes through slot k % slots
    auto send = [&](size_t k) {
        hipError_t e = hipSuccess;
        for (size_t i = batch[k].first; i < batch[k].last && e == hipSuccess; i++)
            e = enqueue(todo[i], ring.buf + (k % slots) * kChunk + todo[i].at, s);
        return e == hipSuccess ? hipEventRecord(ring.ev[k % slots], s) : e;
    };
    auto take = [&](size_t k) {
        const hipError_t e = hipEventSynchronize(ring.ev[k % slots]);
        for (size_t i = batch[k].first; i < batch[k].last && e == hipSuccess; i++)
            std::memcpy(todo[i].dst(), ring.buf + (k % slots) * kChunk + todo[i].at, todo[i].bytes());
        return e;
    };
    hipError_t e = hipSuccess;
    if (alone) {
        for (size_t k = 0; k < slots && e == hipSuccess; k++) e = send(k);
        for (size_t k = 0; k < nb && e == hipSuccess; k++) {
            e = take(k);
            if (e == hipSuccess && k + slots < nb) e = send(k + slots);
        }
        const hipError_t w = hipStreamSynchronize(s);
        return e == hipSuccess ? w : e;
    }

    std::mutex m;
    std::condition_variable arrived, freed;
    size_t queued = 0, next = 0, gone = 0;   // sent; given to a helper; every batch below `gone` has left its slot
    std::vector<char> done(nb, 0);
    bool stop = false;
    hipError_t werr = hipSuccess;
    int dev = 0;
    (void)hipGetDevice(&dev);
    auto work = [&]() {
        (void)hipSetDevice(dev);
        for (;;) {
            size_t k;
            {
                std::unique_lock<std::mutex> l(m);
                arrived.wait(l, [&] { return next < queued || next == nb || stop; });
                if (next >= queued) return;
                k = next++;
            }
            const hipError_t r = take(k);
            {
                std::lock_guard<std::mutex> l(m);
                if (r != hipSuccess) werr = r;
                done[k] = 1;
                while (gone < nb && done[gone]) gone++;
            }
            freed.notify_one();
        }
    };
    std::vector<std::thread> pool;
    const int helpers = (int)std::min<size_t>(kThreads, bytes / kThreadShare);
    pool.reserve(helpers);
    for (int t = 0; t < helpers; t++) {
        try {
            pool.emplace_back(work);
        } catch (...) {
            break;   // fewer helpers
        }
    }
    if (pool.empty()) return deliver_plain(todo, s);
    for (size_t k = 0; k < nb && e == hipSuccess; k++) {
        {
            std::unique_lock<std::mutex> l(m);
            freed.wait(l, [&] { return k < gone + slots; });
        }
        e = send(k);
        if (e == hipSuccess) {
            {
                std::lock_guard<std::mutex> l(m);
                queued = k + 1;
            }
            arrived.notify_one();
        }
    }
    {
        std::lock_guard<std::mutex> l(m);
        stop = e != hipSuccess;
    }
    arrived.notify_all();
    for (std::thread &t : pool) t.join();
    if (e == hipSuccess) e = werr;
    const hipError_t w = hipStreamSynchronize(s);
    return e == hipSuccess ? w : e;
}

}  // namespace pictor
