// The device allocations of the library: counters and kept blocks (devmem.h).
#include "devmem.h"

#include <deque>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace smat {

std::atomic<long long> g_dev_mallocs{0}, g_dev_frees{0}, g_dev_fail_in{-1};

namespace {

struct Block {
    size_t bytes; // of the size class
    int device;
    bool kept; // released by the library, still allocated
};

struct Keeper {
    std::mutex mutex;
    std::unordered_map<void *, Block> blocks; // handed out or kept; larger ones than DEV_KEEP_BLOCK are not listed
    struct PerDevice {
        std::map<size_t, std::vector<void *>> kept; // by size class, the one released last at the back
        std::deque<void *> order;                   // oldest first; entries handed out again are skipped
        size_t bytes = 0;
    };
    std::map<int, PerDevice> devices;
};
Keeper &keeper()
{
    static Keeper *k = new Keeper; // never destroyed: plans of static lifetime may be released after it
    return *k;
}

// eighths of a power of two: at most 12.5 % more than asked for
size_t size_class(size_t bytes)
{
    size_t top = 512;
    while (top < bytes) top <<= 1;
    if (top == 512) return top;
    const size_t step = top / 16;
    return (bytes + step - 1) / step * step;
}

void forget(Keeper::PerDevice &d, size_t bytes, void *p)
{
    std::vector<void *> &v = d.kept[bytes];
    for (size_t i = 0; i < v.size(); i++)
        if (v[i] == p) {
            v.erase(v.begin() + (long)i);
            break;
        }
    d.bytes -= bytes;
}

// Takes kept blocks out of the books, oldest first, until at most `most` bytes are kept; the caller frees them.
std::vector<void *> take_oldest(Keeper &k, Keeper::PerDevice &d, size_t most)
{
    std::vector<void *> out;
    while (d.bytes > most && !d.order.empty()) {
        void *p = d.order.front();
        d.order.pop_front();
        auto it = k.blocks.find(p);
        if (it == k.blocks.end() || !it->second.kept) continue;
        forget(d, it->second.bytes, p);
        k.blocks.erase(it);
        out.push_back(p);
    }
    return out;
}

hipError_t release(void *p, bool idle)
{
    g_dev_frees.fetch_add(1, std::memory_order_relaxed);
    if (!p) return hipSuccess;
    Keeper &k = keeper();
    int device = -1;
    const bool here = hipGetDevice(&device) == hipSuccess;
    {
        std::lock_guard<std::mutex> lock(k.mutex);
        auto it = k.blocks.find(p);
        if (it == k.blocks.end()) idle = true, device = -1; // the driver's business
        else if (it->second.kept) return hipErrorInvalidValue; // released before
        else if (!here || it->second.device != device) k.blocks.erase(it), device = -1;
    }
    if (device < 0) return hipFree(p);
    if (!idle) {
        const hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) return e;
    }
    std::vector<void *> over;
    {
        std::lock_guard<std::mutex> lock(k.mutex);
        auto it = k.blocks.find(p);
        if (it == k.blocks.end() || it->second.kept) return hipErrorInvalidValue;
        Keeper::PerDevice &d = k.devices[device];
        it->second.kept = true;
        d.kept[it->second.bytes].push_back(p);
        d.bytes += it->second.bytes;
        d.order.push_back(p);
        if (d.order.size() > 4096) { // entries of blocks handed out again, or listed twice
            std::deque<void *> live;
            std::unordered_map<void *, bool> seen;
            for (auto o = d.order.rbegin(); o != d.order.rend(); ++o) {
                auto b = k.blocks.find(*o);
                if (b != k.blocks.end() && b->second.kept && !seen[*o]) live.push_front(*o), seen[*o] = true;
            }
            d.order.swap(live);
        }
        over = take_oldest(k, d, DEV_KEEP_BYTES);
    }
    hipError_t e = hipSuccess;
    for (void *q : over) {
        const hipError_t f = hipFree(q);
        if (e == hipSuccess) e = f;
    }
    return e;
}

} // namespace

hipError_t dev_malloc_bytes(void **p, size_t bytes)
{
    *p = nullptr;
    if (g_dev_fail_in.load(std::memory_order_relaxed) >= 0 && g_dev_fail_in.fetch_sub(1) == 0) return hipErrorOutOfMemory;
    g_dev_mallocs.fetch_add(1, std::memory_order_relaxed);
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    const size_t cls = bytes <= DEV_KEEP_BLOCK ? size_class(bytes) : 0;
    Keeper &k = keeper();
    if (cls) {
        std::lock_guard<std::mutex> lock(k.mutex);
        Keeper::PerDevice &d = k.devices[device];
        auto it = d.kept.find(cls);
        if (it != d.kept.end() && !it->second.empty()) {
            *p = it->second.back();
            it->second.pop_back();
            d.bytes -= cls;
            k.blocks[*p].kept = false;
            return hipSuccess;
        }
    }
    e = hipMalloc(p, cls ? cls : bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        dev_trim(false);
        e = hipMalloc(p, cls ? cls : bytes);
    }
    if (e == hipSuccess && cls) {
        std::lock_guard<std::mutex> lock(k.mutex);
        k.blocks[*p] = Block{cls, device, false};
    }
    return e;
}

hipError_t dev_free(void *p) { return release(p, false); }
hipError_t dev_free_idle(void *p) { return release(p, true); }

void dev_trim(bool all_devices)
{
    int device = 0;
    if (!all_devices && hipGetDevice(&device) != hipSuccess) return;
    Keeper &k = keeper();
    std::vector<void *> all;
    {
        std::lock_guard<std::mutex> lock(k.mutex);
        for (auto &d : k.devices) {
            if (!all_devices && d.first != device) continue;
            const std::vector<void *> some = take_oldest(k, d.second, 0);
            all.insert(all.end(), some.begin(), some.end());
            d.second.order.clear();
        }
    }
    for (void *q : all) (void)hipFree(q);
}

} // namespace smat
