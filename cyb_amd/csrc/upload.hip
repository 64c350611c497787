// upload.hip - model load: interchange tensors in host memory -> native tiles in HBM.
//
// Bound by the host link (57 GB/s from pinned memory where this was measured).  The source is pageable - a
// mapped file, whose pages are also touched for the first time here - so somebody has to copy it into pinned memory:
// one thread does that at 29 GB/s, four at 73, and the pages' faults are taken in parallel too.  The repack
// kernel then reads the pinned slots itself: the bytes cross the bus once, coalesced, and leave the kernel as native
// tiles; the wide-scale scan that a host loop used to make over every scale is part of the same pass.  A slot is 4 MiB
// (reads across the bus reach 50 GB/s in pieces of that size, 37 in pieces of 1 MiB), four of them keep copying
// and reading overlapped.  One decoder layer of Q4 blocks (123 MB, seven tensors, warm page cache): 25 ms with a
// pageable hipMemcpy and a host scan per tensor, 2.7 ms with this (46 GB/s).
#include "upload.h"

#include <string.h>

#include <algorithm>
#include <system_error>

#include "cybq_internal.h"

namespace cybq {

namespace {

inline void cpu_pause() { __builtin_ia32_pause(); }

// spins a little, then lets others run: waits here are for tens of microseconds of copying by running threads
struct Backoff {
    int n = 0;
    void wait()
    {
        if (++n < 256) cpu_pause();
        else std::this_thread::yield();
    }
};

size_t row_q_bytes(const UploadItem& it)
{
    const size_t groups = (size_t)(it.K / kGroup);
    if (it.layout == 0) return groups * (it.quant == 4 ? 16 : 32);
    return groups * (it.quant == 4 ? 18 : 34);
}

size_t row_scale_bytes(const UploadItem& it) { return it.layout == 0 ? (size_t)(it.K / kGroup) * 2 : 0; }

}  // namespace

Uploader::~Uploader()
{
    {
        std::lock_guard<std::mutex> lock(m_);
        quit_ = true;
    }
    wake_.notify_all();
    for (std::thread& t : threads_) t.join();
    for (hipEvent_t e : slot_free_)
        if (e) (void)hipEventDestroy(e);
    if (stream_) (void)hipStreamDestroy(stream_);
    if (ring_) (void)hipHostFree(ring_);
    if (flags_) (void)hipHostFree(flags_);
}

hipError_t Uploader::start()
{
    if (started_) return hipSuccess;
    hipError_t e = hipSuccess;
    if (!ring_) e = hipHostMalloc(reinterpret_cast<void**>(&ring_), kSlots * kSlotBytes, hipHostMallocDefault);
    if (e == hipSuccess && !flags_) e = hipHostMalloc(reinterpret_cast<void**>(&flags_), kMaxFlags * sizeof(uint32_t), hipHostMallocDefault);
    if (e == hipSuccess && !stream_) e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking);
    for (hipEvent_t& ev : slot_free_)
        if (e == hipSuccess && !ev) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    // (six threads copy faster than the link takes it; on a small machine leave half of it to others.  A thread that
    // cannot be had is not missed: the caller copies what nobody else does)
    const int want = std::max(1, std::min(6, (int)std::thread::hardware_concurrency() / 2));
    try {
        while ((int)threads_.size() < want) threads_.emplace_back([this] { worker(); });
    } catch (const std::system_error&) {
    }
    started_ = true;
    return hipSuccess;
}

// one tensor -> pieces of whole strips, each piece -> units
void Uploader::cut(const UploadItem& it, int64_t index)
{
    const size_t qb = row_q_bytes(it), sb = row_scale_bytes(it);
    int64_t rows_per = (int64_t)((kSlotBytes - 2 * kScalesAlign) / (qb + sb)) / kTileN * kTileN;
    for (int64_t r = 0; r < it.N; r += rows_per) {
        Piece p;
        p.item = index;
        p.row0 = r;
        p.rows = std::min(rows_per, it.N - r);
        p.scales_off = ((size_t)p.rows * qb + kScalesAlign - 1) & ~(kScalesAlign - 1);
        p.units = 0;
        auto add = [&](const void* base, size_t row_bytes, size_t off) {
            const uint8_t* src = static_cast<const uint8_t*>(base) + (size_t)r * row_bytes;
            const size_t total = (size_t)p.rows * row_bytes;
            for (size_t o = 0; o < total; o += kUnitBytes, p.units++)
                units_.push_back({src + o, off + o, std::min(kUnitBytes, total - o), (int)pieces_.size()});
        };
        add(it.q, qb, 0);
        if (sb) add(it.scales, sb, p.scales_off);
        pieces_.push_back(p);
    }
}

void Uploader::copy_unit(const Unit& u)
{
    memcpy(ring_ + (size_t)(u.piece % kSlots) * kSlotBytes + u.slot_off, u.src, u.bytes);
    done_[(size_t)u.piece].fetch_add(1, std::memory_order_release);
}

void Uploader::copy_units()
{
    for (;;) {
        const int64_t i = next_unit_.fetch_add(1, std::memory_order_relaxed);
        if (i >= (int64_t)units_.size()) return;
        Backoff b;
        while (units_[(size_t)i].piece >= piece_limit_.load(std::memory_order_acquire)) {
            if (stop_.load(std::memory_order_relaxed)) return;
            b.wait();
        }
        copy_unit(units_[(size_t)i]);
    }
}

void Uploader::worker()
{
    int seen = 0;
    std::unique_lock<std::mutex> lock(m_);
    for (;;) {
        wake_.wait(lock, [&] { return quit_ || job_ != seen; });
        if (quit_) return;
        seen = job_;
        lock.unlock();
        copy_units();
        lock.lock();
        if (--busy_ == 0) idle_.notify_all();
    }
}

hipError_t Uploader::run(UploadItem* items, int64_t count)
{
    hipError_t e = start();
    for (int64_t i = 0; i < count && e == hipSuccess;) {
        if ((row_q_bytes(items[i]) + row_scale_bytes(items[i])) * kTileN + 2 * kScalesAlign > kSlotBytes) {
            e = run_whole(items[i++]);           // one strip does not fit a slot (K beyond 430 000)
            continue;
        }
        int64_t n = 1;
        while (i + n < count && n < kMaxFlags &&
               (row_q_bytes(items[i + n]) + row_scale_bytes(items[i + n])) * kTileN + 2 * kScalesAlign <= kSlotBytes)
            n++;
        e = run_some(items + i, n);
        i += n;
    }
    return e;
}

hipError_t Uploader::run_some(UploadItem* items, int64_t count)
{
    pieces_.clear();
    units_.clear();
    size_t total = 0;
    for (int64_t i = 0; i < count; i++) {
        cut(items[i], i);
        flags_[i] = 0u;
        total += (size_t)items[i].N * (row_q_bytes(items[i]) + row_scale_bytes(items[i]));
    }
    const int n = (int)pieces_.size();
    done_ = std::vector<std::atomic<int>>((size_t)n);
    next_unit_.store(0);
    piece_limit_.store(std::min(n, kSlots));
    stop_.store(false);
    const bool threads = total > kInlineBytes && !threads_.empty();
    if (threads) {
        {
            std::lock_guard<std::mutex> lock(m_);
            busy_ = (int)threads_.size();
            job_++;
        }
        wake_.notify_all();
    }

    // issue pieces in order as their copies finish, hand slots back as their kernels finish
    hipError_t e = hipSuccess;
    int issued = 0, freed = 0;
    size_t next_inline = 0;
    Backoff idle;
    while (issued < n && e == hipSuccess) {
        const Piece& p = pieces_[(size_t)issued];
        if (issued - freed == kSlots) {
            e = hipEventSynchronize(slot_free_[freed % kSlots]);
            freed++;
            piece_limit_.store(std::min(n, freed + kSlots), std::memory_order_release);
            continue;
        }
        if (!threads)
            while (next_inline < units_.size() && units_[next_inline].piece <= issued) copy_unit(units_[next_inline++]);
        if (done_[(size_t)issued].load(std::memory_order_acquire) < p.units) {
            idle.wait();
            continue;
        }
        idle.n = 0;
        const UploadItem& it = items[p.item];
        const uint8_t* slot = ring_ + (size_t)(issued % kSlots) * kSlotBytes;
        const int64_t strip0 = p.row0 / kTileN, strips = (p.rows + kTileN - 1) / kTileN;
        e = launch_repack(it.quant, it.layout, true, slot, it.layout == 0 ? slot + p.scales_off : nullptr,
                          it.dst + (size_t)strip0 * it.KT * tile_bytes(it.quant), (int)p.rows, (int)it.K, (int)strips, it.KT,
                          flags_ + p.item, stream_);
        if (e == hipSuccess) e = hipEventRecord(slot_free_[issued % kSlots], stream_);
        issued++;
    }
    if (e != hipSuccess) stop_.store(true);
    if (threads) {
        std::unique_lock<std::mutex> lock(m_);
        idle_.wait(lock, [&] { return busy_ == 0; });
    }
    const hipError_t es = hipStreamSynchronize(stream_);
    if (e == hipSuccess) e = es;
    for (int64_t i = 0; i < count; i++) items[i].wide = flags_[i] != 0u;
    return e;
}

hipError_t Uploader::run_whole(UploadItem& it)
{
    const size_t qb = (size_t)it.N * row_q_bytes(it), sb = (size_t)it.N * row_scale_bytes(it);
    const size_t s_off = (qb + kScalesAlign - 1) & ~(kScalesAlign - 1);
    uint8_t* tmp = nullptr;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&tmp), s_off + sb + kScalesAlign);
    if (e != hipSuccess) return e;
    flags_[0] = 0u;
    e = hipMemcpy(tmp, it.q, qb, hipMemcpyHostToDevice);
    if (e == hipSuccess && sb) e = hipMemcpy(tmp + s_off, it.scales, sb, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = launch_repack(it.quant, it.layout, false, tmp, sb ? tmp + s_off : nullptr, it.dst, (int)it.N, (int)it.K, it.NT, it.KT, flags_, stream_);
    const hipError_t es = hipStreamSynchronize(stream_);
    if (e == hipSuccess) e = es;
    it.wide = flags_[0] != 0u;
    (void)hipFree(tmp);
    return e;
}

}  // namespace cybq
