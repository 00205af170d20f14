// lv_copy.h -- large copies from the device to the caller's pageable memory.
//
// The runtime copies pageable memory piece by piece on the calling thread, and most of the time of a
// read-out into fresh arrays is that thread's page faults (54 MB: 5.3 ms of a transfer of 1.0).  Here the pieces
// go through a ring of pinned buffers and a few threads, which live as long as the copy, move them on.  Pieces
// end at multiples of 2 MiB of the caller's addresses, so that no two threads fault the same huge page.  A mesh of
// 250,000 particles (54 MB) takes 2.4 ms for 5.3.  Of one field, into memory already touched: 16 MB 0.57 ms for 0.93, 8 MB
// 0.35 for 0.47, 5 MB 0.26 for 0.29, 3 MB 0.18 for 0.19, 2.5 MB 0.16 for 0.15, 2 MB 0.14 for 0.12: copies below 3 MiB
// stay the runtime's, and so do copies to the device (3.2 MB 0.15 ms longer this way).
#pragma once

#include "lv_internal.h"

#include <atomic>
#include <thread>

constexpr int LV_RING = 8;
constexpr size_t LV_PIECE = (size_t)2 << 20;
constexpr int LV_COPIERS = 4;                       // threads at most, one for each MiB (6 and more are no faster)
constexpr size_t LV_STAGED_MIN = (size_t)3 << 20;

// the pinned ring of a context (16 MiB, made by its first large copy)
struct lv_ring {
    char *pin[LV_RING];
    hipEvent_t ev[LV_RING];
    bool made;
};
void lv_ring_free(lv_ring *R);

// One copy operation of about `total` bytes: pushes, then finish, which synchronises the stream; the destinations are
// complete then.
class lv_copier {
  public:
    lv_copier(lv_ring *R, hipStream_t s, size_t total);
    ~lv_copier();
    hipError_t to_host(void *dst, const void *src, size_t bytes);
    hipError_t finish();

  private:
    struct task {
        char *dst;
        const char *src;
        size_t bytes;
    };
    void work();
    void publish();
    hipError_t arrive(unsigned must);  // publishes the pieces that have arrived, having waited for those below `must`
    hipError_t slot_free(unsigned k);

    lv_ring *R;
    hipStream_t s;
    bool staged;
    int nthreads = 0;
    std::thread th[LV_COPIERS];
    task ring[LV_RING] = {};
    std::atomic<unsigned> published{0}, claimed{0};
    std::atomic<bool> busy[LV_RING] = {}, stop{false};
    unsigned issued = 0;
};
