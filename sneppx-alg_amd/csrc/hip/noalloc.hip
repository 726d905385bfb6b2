// noalloc.hip - the scratch buffer of the allocation-free entry point
// (SNEPPX_qlinear_w4a16_noalloc): a file-scope device array of
// SNEPPX_NOALLOC_SCRATCH_BYTES that every GPU the library runs on holds until
// the process ends, so a call needs no device allocation at all.
//
// In host code the array's name is a host-side stand-in, not a device
// address.  Its address on a device comes from hipGetSymbolAddress, looked up
// once per device (with that device current, at the entry point's first call
// there) and kept in known[dev]; only that pointer is ever handed to
// kernels.  Each device has its own copy at its own address.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>

#include "launch.h"
#include "sneppx_qlinear.h"
#include "../snx_internal.h"

static __device__ __align__(256) uint8_t scratch[SNEPPX_NOALLOC_SCRATCH_BYTES];

// Arrival counters of the K spans (zero when the library loads; every call
// leaves them zero), apart from the scratch so that no other call writes them.
// Calls that overlap, against the header's rule, can leave them otherwise, which
// SNEPPX_qlinear_noalloc_reset mends.  (A fill ahead of every call would too: a
// launch more, 11.1 -> 12.9 us at N = 6144, K = 4096, M = 32, and 8.5 -> 11.3 for
// the smallest, which the host's launches bound.)
constexpr size_t kCounterBytes = 64 << 10;
static __device__ __align__(256) uint32_t counters[kCounterBytes / sizeof(uint32_t)];

namespace {
std::atomic<void*> g_scratch[snx::kMaxDevices], g_counters[snx::kMaxDevices];
std::mutex g_scratch_mu;

void* static_array(const void* symbol, std::atomic<void*>* known, size_t bytes, size_t most, const char* who) {
    if (bytes > most) {
        snx_set_error("%s: this call needs %zu bytes of scratch, more than the %zu of the "
                      "library's static buffer", who, bytes, most);
        return nullptr;
    }
    const int dev = snx::current_device();
    if (dev < 0) {
        snx_set_error("%s: no current device (or device index beyond %d)", who, snx::kMaxDevices - 1);
        return nullptr;
    }
    void* p = known[dev].load(std::memory_order_acquire);
    if (p) return p;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = known[dev].load(std::memory_order_relaxed);
    if (!p) {
        const hipError_t e = hipGetSymbolAddress(&p, symbol);
        if (e != hipSuccess || !p) {
            snx_set_error("%s: hipGetSymbolAddress on device %d: %s", who, dev,
                          hipGetErrorString(e));
            return nullptr;
        }
        known[dev].store(p, std::memory_order_release);
    }
    return p;
}
}  // namespace

extern "C" {

void* snx_noalloc_scratch(size_t bytes, const char* who) {
    return static_array(HIP_SYMBOL(scratch), g_scratch, bytes, SNEPPX_NOALLOC_SCRATCH_BYTES, who);
}

void* snx_noalloc_counters(size_t bytes, const char* who) {
    return static_array(HIP_SYMBOL(counters), g_counters, bytes, kCounterBytes, who);
}

int SNEPPX_qlinear_noalloc_reset(SNEPPXStream stream) {
    snx_clear_error();
    void* const cnt = snx_noalloc_counters(kCounterBytes, "qlinear_noalloc_reset");
    return cnt ? snx_k_fill_zero(cnt, kCounterBytes, stream) : -1;
}

}  // extern "C"
