// pool.hip - see pool.h.  Host code only.  Callers have made `device` current.  The containers allocate, and these functions are
// called from C entries: what they throw ends here, as hipErrorOutOfMemory or as a block or slot that is not kept.
#include "pool.h"

#include <deque>
#include <list>
#include <map>
#include <mutex>
#include <new>

namespace cybq {

namespace {

constexpr size_t kGrain = (size_t)64 << 10;             // blocks are multiples of it
constexpr size_t kScanWords = 1024;                     // pinned words per slab
constexpr size_t kScanPitch = 16;                       // (words of different tensors on different host cache lines)

struct Block {
    void* p;
    size_t bytes;
    UsedOn used_on;
};

struct DevicePool {
    std::mutex m;
    int contexts = 0;
    std::list<Block> blocks;                            // oldest first
    size_t held = 0;
    std::deque<ScanSlot> scans;                         // free slots, the longest free first (their pinned memory is kept for the process)
};

DevicePool& pool_of(int device)
{
    static std::mutex m;
    static std::map<int, DevicePool>* pools = new std::map<int, DevicePool>();      // (never destroyed: handles may be freed at exit)
    std::lock_guard<std::mutex> lock(m);
    return (*pools)[device];
}

hipError_t empty(DevicePool& pool)                      // pool.m held
{
    hipError_t first = hipSuccess;
    for (const Block& b : pool.blocks) {
        const hipError_t e = hipFree(b.p);
        if (first == hipSuccess) first = e;
    }
    pool.blocks.clear();
    pool.held = 0;
    return first;
}

}  // namespace

hipError_t pool_retain(int device)
try {
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    pool.contexts++;
    return hipSuccess;
} catch (const std::bad_alloc&) {
    return hipErrorOutOfMemory;
}

void pool_release(int device)
{
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    if (--pool.contexts == 0) (void)empty(pool);
}

hipError_t pool_alloc(int device, size_t bytes, UsedOn first_use, void** p, size_t* block)
{
    bytes = (bytes + kGrain - 1) / kGrain * kGrain;
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    // the smallest block that holds it, if that wastes no more than a quarter
    auto best = pool.blocks.end();
    for (auto it = pool.blocks.begin(); it != pool.blocks.end(); ++it)
        if (it->bytes >= bytes && it->bytes - bytes <= bytes / 4 && (best == pool.blocks.end() || it->bytes < best->bytes)) best = it;
    if (best != pool.blocks.end()) {
        const bool ordered = best->used_on == kUnused || (best->used_on == kDefaultStream && first_use == kDefaultStream);
        if (!ordered) {
            const hipError_t e = hipDeviceSynchronize();
            if (e != hipSuccess) return e;
            for (Block& b : pool.blocks) b.used_on = kUnused;
        }
        *p = best->p;
        *block = best->bytes;
        pool.held -= best->bytes;
        pool.blocks.erase(best);
        return hipSuccess;
    }
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory && !pool.blocks.empty()) {
        (void)hipGetLastError();
        (void)empty(pool);
        e = hipMalloc(p, bytes);
    }
    *block = bytes;
    return e;
}

void pool_free(int device, void* p, size_t block, UsedOn used_on)
{
    if (!p) return;
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    if (pool.contexts == 0 || block > kPoolBytes) {
        (void)hipFree(p);
        return;
    }
    try {
        pool.blocks.push_back({p, block, used_on});
    } catch (const std::bad_alloc&) {
        (void)hipFree(p);
        return;
    }
    pool.held += block;
    while (pool.held > kPoolBytes) {
        (void)hipFree(pool.blocks.front().p);
        pool.held -= pool.blocks.front().bytes;
        pool.blocks.pop_front();
    }
}

hipError_t pool_trim(int device)
{
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    return empty(pool);
}

hipError_t scan_acquire(int device, ScanSlot* s)
try {
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    if (pool.scans.empty()) {
        void* slab = nullptr;
        std::deque<ScanSlot> fresh(kScanWords);
        hipError_t e = hipHostMalloc(&slab, kScanWords * kScanPitch * sizeof(uint32_t), hipHostMallocDefault);
        if (e != hipSuccess) return e;
        for (size_t i = 0; i < kScanWords; i++) fresh[i].word = static_cast<uint32_t*>(slab) + i * kScanPitch;
        pool.scans.swap(fresh);
    }
    ScanSlot& got = pool.scans.front();
    // (events are made as slots are first used, and stay with them; a slot given back ahead of its kernel is waited for)
    const hipError_t e = got.done ? hipEventSynchronize(got.done) : hipEventCreateWithFlags(&got.done, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    *s = got;
    pool.scans.pop_front();
    return hipSuccess;
} catch (const std::bad_alloc&) {
    return hipErrorOutOfMemory;
}

void scan_release(int device, ScanSlot s)
{
    if (!s.word) return;
    DevicePool& pool = pool_of(device);
    std::lock_guard<std::mutex> lock(pool.m);
    try {
        pool.scans.push_back(s);
    } catch (const std::bad_alloc&) {
    }
}

}  // namespace cybq
