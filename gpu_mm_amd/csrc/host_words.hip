// A few words of device memory brought to the host at the end of a call: error flags, counts.

#include <immintrin.h>

#include <atomic>
#include <chrono>
#include <mutex>
#include <vector>

#include "gmm_internal.hpp"

namespace gmm {

namespace {

// A slot of pinned host memory: up to SLOT_WORDS - 1 words and the ticket of the call that wrote them.
constexpr int SLOT_WORDS = 16;                // 64 bytes
constexpr int NSLOTS = 64;                    // one page; each is in use by one call at a time
constexpr int PB_THREADS = 256;
constexpr int PB_LOADS = 16;                  // in flight per thread (a call with 262144 error words 907 -> 620 us)

// Stores n words of src (their OR, when 'any') and then the ticket, where the host sees them. One block;
// it runs after everything that was enqueued on its stream before it.
__global__ void __launch_bounds__(PB_THREADS)
publish_words_kernel(const uint32_t *__restrict__ src, int64_t n, bool any, uint32_t *slot, uint32_t ticket)
{
    __shared__ uint32_t s_or;
    uint32_t v = 0;
    if (any) {
        if (threadIdx.x == 0)
            s_or = 0;
        __syncthreads();
        for (int64_t i0 = 0; i0 < n; i0 += PB_THREADS * PB_LOADS) {
            uint32_t w[PB_LOADS];
#pragma unroll
            for (int k = 0; k < PB_LOADS; k++) {
                const int64_t i = i0 + k * PB_THREADS + threadIdx.x;
                w[k] = (i < n) ? src[i] : 0u;
            }
#pragma unroll
            for (int k = 0; k < PB_LOADS; k++)
                v |= w[k];
        }
        if (v)
            atomicOr(&s_or, v);
        __syncthreads();
        v = s_or;
        n = 1;
    }
    else if (threadIdx.x < n)
        v = src[threadIdx.x];
    if (threadIdx.x < n)
        __hip_atomic_store(slot + threadIdx.x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(slot + SLOT_WORDS - 1, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The slots not in use. Allocated at the first call and kept until the process ends.
class Slots
{
public:
    uint32_t *take()
    {
        std::lock_guard<std::mutex> lk(mu);
        if (!page && !failed) {
            void *p = nullptr;
            // Allowed while a stream of this thread captures: nothing is enqueued.
            hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
            (void)hipThreadExchangeStreamCaptureMode(&mode);
            failed = hipHostMalloc(&p, NSLOTS * SLOT_WORDS * 4,
                                   hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess;
            (void)hipThreadExchangeStreamCaptureMode(&mode);
            if (failed)
                (void)hipGetLastError();
            else {
                page = static_cast<uint32_t *>(p);
                for (int i = 0; i < NSLOTS; i++) {
                    page[i * SLOT_WORDS + SLOT_WORDS - 1] = 0;
                    free_slots.push_back(page + i * SLOT_WORDS);
                }
            }
        }
        if (free_slots.empty())
            return nullptr;
        uint32_t *s = free_slots.back();
        free_slots.pop_back();
        return s;
    }

    void give_back(uint32_t *s)
    {
        std::lock_guard<std::mutex> lk(mu);
        free_slots.push_back(s);                   // capacity for NSLOTS is there since take()
    }

private:
    std::mutex mu;
    uint32_t *page = nullptr;
    bool failed = false;
    std::vector<uint32_t *> free_slots;
};

Slots &slots()
{
    static Slots *s = new Slots;                   // never destroyed: calls may come from any thread, to the end
    return *s;
}

void copy_words(uint32_t *out, const uint32_t *src, int64_t n, bool any, hipStream_t stream)
{
    std::vector<uint32_t> h(static_cast<size_t>(n), 0u);
    GMM_HIP(hipMemcpyAsync(h.data(), src, size_t(n) * 4, hipMemcpyDeviceToHost, stream));
    GMM_HIP(hipStreamSynchronize(stream));
    if (any) {
        *out = 0;
        for (uint32_t v : h)
            *out |= v;
    }
    else
        std::copy(h.begin(), h.end(), out);
}

// The host waits for the ticket that a one-block kernel stores in pinned memory after the words, instead
// of copying 4 bytes to pageable memory and waiting for the stream: 11 us less a call (map2tod and tod2map
// of 8 x 4096 samples with their checks 87.6 -> 65.6 us, preplan and plan of 7 x 4099 136 -> 90 us). After
// SPIN_US the wait goes to hipStreamSynchronize(), which also reports a failed stream. A capturing stream
// takes the copy, which refuses it.
constexpr int SPIN_US = 200;

void fetch(uint32_t *out, const uint32_t *src, int64_t n, bool any, hipStream_t stream)
{
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    uint32_t *slot = nullptr;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess)
        (void)hipGetLastError();
    else if (cap == hipStreamCaptureStatusNone && (any || n < SLOT_WORDS))
        slot = slots().take();
    if (!slot)
        return copy_words(out, src, n, any, stream);

    // An error from here on keeps the slot out of use: a kernel may still write it.
    volatile uint32_t *done = slot + SLOT_WORDS - 1;
    const uint32_t ticket = *done + 1;
    publish_words_kernel<<<1, PB_THREADS, 0, stream>>>(src, n, any, slot, ticket);
    GMM_HIP(hipGetLastError());
    const auto t0 = std::chrono::steady_clock::now();
    while (*done != ticket) {
        for (int i = 0; i < 16 && *done != ticket; i++)
            _mm_pause();
        if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(SPIN_US)) {
            GMM_HIP(hipStreamSynchronize(stream));
            break;
        }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    for (int64_t i = 0; i < (any ? 1 : n); i++)
        out[i] = const_cast<volatile uint32_t *>(slot)[i];
    slots().give_back(slot);
}

}  // namespace

void read_words(uint32_t *out, const uint32_t *src, int n, hipStream_t stream) { fetch(out, src, n, false, stream); }

uint32_t read_word(const uint32_t *p, hipStream_t stream)
{
    uint32_t h = 0;
    read_words(&h, p, 1, stream);
    return h;
}

uint32_t read_word_of_any_device(const uint32_t *p)
{
    // A kernel of the current device may not be able to read another device's memory; a copy can.
    int dev = 0;
    hipPointerAttribute_t attr = {};
    if (hipGetDevice(&dev) == hipSuccess && hipPointerGetAttributes(&attr, p) == hipSuccess && attr.device == dev)
        return read_word(p, nullptr);
    (void)hipGetLastError();
    uint32_t h = 0;
    copy_words(&h, p, 1, false, nullptr);
    return h;
}

uint32_t read_word_or(const uint32_t *p, int64_t n, hipStream_t stream)
{
    uint32_t h = 0;
    fetch(&h, p, n, true, stream);
    return h;
}

}  // namespace gmm
