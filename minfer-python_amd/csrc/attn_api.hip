// Entry points of the C ABI that are not tied to one operator.
#include <mutex>

#include "attn_host.h"

namespace minfer_attn {
static __device__ uint32_t counter_pool[kCounterStreams * kStreamCounters];   // zero when the code object is loaded

uint32_t* stream_counters(hipStream_t stream) {
    if (stream == hipStreamPerThread) return nullptr;   // one handle, another stream in every thread
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &st) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    if (st != hipStreamCaptureStatusNone) return nullptr;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    struct Device { uint32_t* base = nullptr; int n = 0; hipStream_t stream[kCounterStreams]; };
    static std::mutex mu;
    static Device devices[64];
    std::lock_guard<std::mutex> lock(mu);
    Device& d = devices[dev];
    for (int i = 0; i < d.n; ++i)
        if (d.stream[i] == stream) return d.base + (size_t)i * kStreamCounters;
    if (d.n == kCounterStreams) return nullptr;
    if (!d.base) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(counter_pool)) != hipSuccess || !ptr) { (void)hipGetLastError(); return nullptr; }
        d.base = (uint32_t*)ptr;
    }
    d.stream[d.n] = stream;
    return d.base + (size_t)d.n++ * kStreamCounters;
}
}  // namespace minfer_attn

MINFER_ATTN_EXPORT int minfer_attn_version(void) { return 1000; }

MINFER_ATTN_EXPORT const char* minfer_attn_last_error(void) { return minfer_attn::error_buf(); }
