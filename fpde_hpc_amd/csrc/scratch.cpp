// Device scratch memory of the calls that need some for their duration (the
// direct history sums and GEMMs, the facade's "Sum"): a hipMalloc/hipFree
// pair per call costs more than the kernels of a small one (hipFree waits for
// the device), and for a large one milliseconds of mapping.
//
// Buffers are leased: while a lease lives nobody else has its buffer, and its
// owner gives it back only when the device has finished with it, so a buffer
// is never shared between threads or streams.  Returned buffers are kept for
// the next lease on their device up to kPoolBytes in all, the rest is freed;
// an allocation of the library that the device refuses frees what its pool
// keeps and tries again (device_malloc), and fpde_shutdown frees every buffer
// that is not leased.
#include "fpde_internal.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <new>

namespace fpde {

namespace {
constexpr size_t kPoolBytes = (size_t)256 << 20;      // kept per device
struct DevicePool {
    std::multimap<size_t, void*> free;                // by size
    size_t held = 0;
};
std::mutex g_pool_mu;
std::map<int, DevicePool> g_pool;
}  // namespace

// Frees what the pool keeps on the current device; whether that was anything.
static bool trim_pool() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lock(g_pool_mu);
    const auto pool = g_pool.find(dev);
    if (pool == g_pool.end() || pool->second.free.empty()) return false;
    for (auto& b : pool->second.free) (void)hipFree(b.second);
    pool->second.free.clear();
    pool->second.held = 0;
    return true;
}

hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess && trim_pool()) e = hipMalloc(p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();     // reported here, not by the next call
    return e;
}

fpde_status ScratchLease::take(size_t bytes, int device, size_t at_most) {
    give();
    int cur = 0;
    FPDE_HIP_TRY(hipGetDevice(&cur));
    const int dev = device < 0 ? cur : device;
    const size_t want = std::max<size_t>((bytes + 0xfffff) & ~(size_t)0xfffff, (size_t)1 << 20);
    {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        DevicePool& p = g_pool[dev];
        auto it = p.free.lower_bound(want);
        if (it != p.free.end() && it->first <= std::max(at_most, want)) {
            bytes_ = it->first;
            ptr_ = it->second;
            p.held -= it->first;
            p.free.erase(it);
            dev_ = dev;
            return FPDE_OK;
        }
    }
    void* q = nullptr;
    if (dev != cur) FPDE_HIP_TRY(hipSetDevice(dev));
    const hipError_t e = device_malloc(&q, want);
    if (dev != cur) (void)hipSetDevice(cur);
    if (e != hipSuccess) {
        set_error(std::string("scratch memory: ") + hipGetErrorString(e));
        return FPDE_ERR_NOMEM;
    }
    ptr_ = q;
    bytes_ = want;
    dev_ = dev;
    return FPDE_OK;
}

void ScratchLease::give() {
    if (!ptr_) return;
    void* q = ptr_;
    ptr_ = nullptr;
    try {
        std::lock_guard<std::mutex> lock(g_pool_mu);
        DevicePool& p = g_pool[dev_];
        if (p.held + bytes_ <= kPoolBytes) {
            p.free.emplace(bytes_, q);
            p.held += bytes_;
            return;
        }
    } catch (const std::bad_alloc&) {                 // no room for its entry: not kept (destructors come here)
    }
    (void)hipFree(q);
}

bool scratch_shutdown() {
    std::lock_guard<std::mutex> lock(g_pool_mu);
    bool ok = true;
    for (auto& d : g_pool) {
        for (auto& b : d.second.free) ok = hipFree(b.second) == hipSuccess && ok;
        d.second.free.clear();
        d.second.held = 0;
    }
    return ok;
}

}  // namespace fpde
