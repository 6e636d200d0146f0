// Every device allocation of the library goes through these, so that one pair of counters says how many
// there were: the test of the entry point that allocates nothing reads them (smat_internal_alloc_counts).
//
// Released blocks are kept for the next allocation of their size class instead of going back to the driver: a
// hipMalloc / hipFree pair costs 10 us for a few bytes and several hundred for the 121 MB of blocks of a 16384^2
// matrix, and blocking, planning and looking at the values of one new matrix makes thirty of them.  What is kept is
// bounded (DEV_KEEP_BYTES per device, blocks of at most DEV_KEEP_BLOCK), goes back to the driver oldest first when
// the bound is reached, and altogether when an allocation fails or smat_plan_cache_clear is called.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

namespace smat {
extern std::atomic<long long> g_dev_mallocs, g_dev_frees;
extern std::atomic<long long> g_dev_fail_in; // test hook: so many allocations from now on succeed, the next fails; < 0: none

constexpr size_t DEV_KEEP_BYTES = (size_t)1 << 30, DEV_KEEP_BLOCK = (size_t)1 << 29;

hipError_t dev_malloc_bytes(void **p, size_t bytes);
template <class T> inline hipError_t dev_malloc(T **p, size_t bytes)
{
    return dev_malloc_bytes(reinterpret_cast<void **>(p), bytes);
}
// Waits for the work on the device, as hipFree does: nothing may still use a block that the next allocation gets.
hipError_t dev_free(void *p);
// The same for a caller that has waited since the last use of the block.
hipError_t dev_free_idle(void *p);
// Gives the kept blocks, of the current device or of all, back to the driver.
void dev_trim(bool all_devices);

// Scratch memory of one call.  Its release waits for the device (some 18 us behind a copy to the host) unless the call says that it has
// waited since the last use.
struct DevScratch {
    void *p = nullptr;
    bool idle = false;
    DevScratch() = default;
    DevScratch(const DevScratch &) = delete;
    DevScratch &operator=(const DevScratch &) = delete;
    ~DevScratch() { release(); }
    void release()
    {
        if (p) (void)(idle ? dev_free_idle(p) : dev_free(p));
        p = nullptr;
    }
    hipError_t alloc(size_t bytes)
    {
        idle = false;
        return dev_malloc(&p, bytes ? bytes : 16);
    }
};
} // namespace smat
