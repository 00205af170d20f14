// lv_copy.hip -- large copies from the device to pageable memory (lv_copy.h).  Host code.
#include "lv_copy.h"

#include <algorithm>
#include <cstring>

#define COPY_CHECK(expr)                 \
    do {                                 \
        hipError_t _e = (expr);          \
        if (_e != hipSuccess) return _e; \
    } while (0)

static bool ring_make(lv_ring *R)
{
    if (R->made) return true;
    for (int k = 0; k < LV_RING; k++) {
        if (!R->pin[k] && hipHostMalloc((void **)&R->pin[k], LV_PIECE, hipHostMallocDefault) != hipSuccess) {
            R->pin[k] = nullptr;
            (void)hipGetLastError();
            return false;
        }
        if (!R->ev[k] && hipEventCreateWithFlags(&R->ev[k], hipEventDisableTiming) != hipSuccess) {
            R->ev[k] = nullptr;
            (void)hipGetLastError();
            return false;
        }
    }
    R->made = true;
    return true;
}

void lv_ring_free(lv_ring *R)
{
    for (int k = 0; k < LV_RING; k++) {
        if (R->pin[k]) (void)hipHostFree(R->pin[k]);
        if (R->ev[k]) (void)hipEventDestroy(R->ev[k]);
        R->pin[k] = nullptr;
        R->ev[k] = nullptr;
    }
    R->made = false;
}

lv_copier::lv_copier(lv_ring *R_, hipStream_t s_, size_t total) : R(R_), s(s_)
{
    staged = total >= LV_STAGED_MIN && ring_make(R);  // (without the pinned memory: the runtime's copies)
    if (!staged) return;
    const int want = (int)std::min<size_t>(LV_COPIERS, total >> 20);
    try {
        for (; nthreads < want; nthreads++) th[nthreads] = std::thread(&lv_copier::work, this);
    } catch (...) {  // as many as there are; none: the calling thread moves the pieces
    }
}

lv_copier::~lv_copier()
{
    stop.store(true, std::memory_order_release);
    for (int k = 0; k < nthreads; k++) th[k].join();
}

void lv_copier::work()
{
    for (;;) {
        unsigned k = claimed.load(std::memory_order_relaxed);
        // (not == : a claim of another thread may be seen before the piece it claimed is)
        if ((int)(published.load(std::memory_order_acquire) - k) <= 0) {
            if (stop.load(std::memory_order_acquire)) return;
            std::this_thread::yield();
            continue;
        }
        if (!claimed.compare_exchange_weak(k, k + 1, std::memory_order_relaxed)) continue;
        const task t = ring[k % LV_RING];
        memcpy(t.dst, t.src, t.bytes);
        busy[k % LV_RING].store(false, std::memory_order_release);
    }
}

// the task in the slot of `published` is ready
void lv_copier::publish()
{
    const unsigned k = published.load(std::memory_order_relaxed), q = k % LV_RING;
    if (nthreads == 0) {
        memcpy(ring[q].dst, ring[q].src, ring[q].bytes);
        busy[q].store(false, std::memory_order_relaxed);
        claimed.store(k + 1, std::memory_order_relaxed);
    }
    published.store(k + 1, std::memory_order_release);
}

hipError_t lv_copier::arrive(unsigned must)
{
    while (published.load(std::memory_order_relaxed) != issued) {
        const unsigned k = published.load(std::memory_order_relaxed), q = k % LV_RING;
        if (k < must) {
            COPY_CHECK(hipEventSynchronize(R->ev[q]));
        } else {
            const hipError_t e = hipEventQuery(R->ev[q]);
            if (e == hipErrorNotReady) return hipSuccess;
            COPY_CHECK(e);
        }
        publish();
    }
    return hipSuccess;
}

hipError_t lv_copier::slot_free(unsigned k)
{
    while (busy[k % LV_RING].load(std::memory_order_acquire)) {
        COPY_CHECK(arrive(k - LV_RING + 1));
        std::this_thread::yield();
    }
    return hipSuccess;
}

hipError_t lv_copier::to_host(void *dst, const void *src, size_t bytes)
{
    if (!staged) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    char *d = (char *)dst;
    const char *p = (const char *)src;
    while (bytes > 0) {
        const size_t m = std::min(bytes, LV_PIECE - ((uintptr_t)d & (LV_PIECE - 1)));
        COPY_CHECK(slot_free(issued));
        const unsigned q = issued % LV_RING;
        busy[q].store(true, std::memory_order_relaxed);
        ring[q] = task{d, R->pin[q], m};
        COPY_CHECK(hipMemcpyAsync(R->pin[q], p, m, hipMemcpyDeviceToHost, s));
        COPY_CHECK(hipEventRecord(R->ev[q], s));
        issued++;
        COPY_CHECK(arrive(0));
        d += m;
        p += m;
        bytes -= m;
    }
    return hipSuccess;
}

hipError_t lv_copier::finish()
{
    if (staged) {
        COPY_CHECK(arrive(issued));
        for (unsigned q = 0; q < LV_RING; q++)
            while (busy[q].load(std::memory_order_acquire)) std::this_thread::yield();
    }
    return hipStreamSynchronize(s);
}
