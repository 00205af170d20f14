// lv_mail.hip -- a few device integers to the host without a copy and a stream synchronisation.
//
// A kernel of one wavefront copies them to pinned host memory behind everything launched before it and
// then stores the number of the request, for which the host spins: some 10 us sooner than an
// asynchronous copy and a synchronisation, and the host can launch more work between post and await.
#include "lv_internal.h"

#include <chrono>
#include <cstring>

namespace {

__global__ __launch_bounds__(64) void k_mail(int *__restrict__ src, int cnt, int nclear, int *__restrict__ dst, int seq)
{
    const int t = threadIdx.x;
    if (t < cnt) {
        dst[1 + t] = src[t];
        if (t < nclear) src[t] = 0;
        __threadfence_system();
    }
    __syncthreads();
    if (t == 0) __hip_atomic_store(dst, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

hipError_t lv_mail_init(lv_mailbox *mb)
{
    const size_t bytes = sizeof(int) * (1 + LV_MAIL_MAX);
    hipError_t e = hipHostMalloc((void **)&mb->host, bytes, hipHostMallocCoherent | hipHostMallocMapped);
    if (e != hipSuccess) {
        mb->host = nullptr;
        return e;
    }
    memset(mb->host, 0, bytes);
    mb->seq = 0;
    e = hipHostGetDevicePointer((void **)&mb->dev, mb->host, 0);
    if (e != hipSuccess) lv_mail_free(mb);
    return e;
}

void lv_mail_free(lv_mailbox *mb)
{
    if (mb->host) (void)hipHostFree(mb->host);
    mb->host = mb->dev = nullptr;
}

hipError_t lv_mail_post(lv_mailbox *mb, int *src, int cnt, int nclear, hipStream_t s)
{
    if (cnt > LV_MAIL_MAX || nclear > cnt) return hipErrorInvalidValue;
    mb->seq = mb->seq == 0x7fffffff ? 1 : mb->seq + 1;
    hipLaunchKernelGGL(k_mail, dim3(1), dim3(64), 0, s, src, cnt, nclear, mb->dev, mb->seq);
    return hipGetLastError();
}

hipError_t lv_mail_await(lv_mailbox *mb, int *out, int cnt, hipStream_t s)
{
    const auto t0 = std::chrono::steady_clock::now();
    for (int spin = 1; __atomic_load_n(mb->host, __ATOMIC_ACQUIRE) != mb->seq; spin++) {
        if ((spin & 255) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(20)) {
            hipError_t e = hipStreamSynchronize(s);
            if (e != hipSuccess) return e;
            if (__atomic_load_n(mb->host, __ATOMIC_ACQUIRE) != mb->seq) return hipErrorUnknown;
        }
    }
    memcpy(out, mb->host + 1, sizeof(int) * cnt);
    return hipSuccess;
}
