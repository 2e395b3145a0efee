// Entry points of the C ABI that are not tied to one operator.
#include <atomic>

#include "attn_host.h"

namespace minfer_attn {
static __device__ uint32_t counter_pool[kStreamCounters];   // zero when the code object is loaded, on every device

uint32_t* stream_counters(hipStream_t stream) {
    if (stream) return nullptr;
    static std::atomic<uint32_t*> base[64];   // concurrent first calls at worst both look the address up
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { (void)hipGetLastError(); return nullptr; }
    uint32_t* p = base[dev].load(std::memory_order_acquire);
    if (!p) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(counter_pool)) != hipSuccess || !ptr) { (void)hipGetLastError(); return nullptr; }
        p = (uint32_t*)ptr;
        base[dev].store(p, std::memory_order_release);
    }
    return p;
}
}  // namespace minfer_attn

MINFER_ATTN_EXPORT int minfer_attn_version(void) { return 1000; }

MINFER_ATTN_EXPORT const char* minfer_attn_last_error(void) { return minfer_attn::error_buf(); }
