// upload.h - host memory -> native weights: the engine behind cybq_weight_upload / cybq_weight_upload_many.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace cybq {

// one tensor on its way from host memory to its native tiles (destination allocated by the caller)
struct UploadItem {
    int quant, layout;
    int64_t N, K;
    const void *q, *scales;
    uint8_t* dst;
    int NT, KT;
    bool wide = false;               // result: some |scale| times the largest |q| leaves f16
};

// A context's upload engine.  Source buffers are pageable memory (the mapped model file): they are copied by a few
// threads into a ring of pinned slots, and the repack kernel reads the slots across the bus itself - no staging
// buffer on the device and no second pass there.  A slot holds whole 16-row strips.  Everything is created by the first
// upload and kept until the context goes: the ring is 16 MiB of pinned memory, the threads sleep in between.
class Uploader {
public:
    Uploader() = default;
    Uploader(const Uploader&) = delete;
    Uploader& operator=(const Uploader&) = delete;
    ~Uploader();
    // Returns when the source buffers have been read and every tensor is in place.
    hipError_t run(UploadItem* items, int64_t count);

private:
    static constexpr int kSlots = 4;
    static constexpr size_t kSlotBytes = (size_t)4 << 20;
    static constexpr size_t kUnitBytes = (size_t)256 << 10;      // what a thread copies at a time
    static constexpr size_t kInlineBytes = (size_t)512 << 10;    // jobs up to this size are copied by the caller
    static constexpr size_t kScalesAlign = 256;
    static constexpr int kMaxFlags = 1024;                        // tensors per pass over the ring

    struct Piece {                   // consecutive strips of one tensor that share a slot
        int64_t item, row0, rows;
        size_t scales_off;           // PLANAR: where in the slot the scales start
        int units;
    };
    struct Unit {                    // one memcpy into a slot
        const uint8_t* src;
        size_t slot_off, bytes;
        int piece;
    };

    hipError_t start();
    hipError_t run_some(UploadItem* items, int64_t count);
    hipError_t run_whole(UploadItem& it);
    void cut(const UploadItem& it, int64_t index);
    void copy_unit(const Unit& u);
    void copy_units();
    void worker();

    bool started_ = false;
    uint8_t* ring_ = nullptr;
    uint32_t* flags_ = nullptr;      // pinned: a repack kernel that meets a wide scale stores 1 in its tensor's word
    hipStream_t stream_ = nullptr;
    hipEvent_t slot_free_[kSlots] = {};
    std::vector<Piece> pieces_;
    std::vector<Unit> units_;
    std::vector<std::atomic<int>> done_;          // units of a piece that have been copied
    std::atomic<int64_t> next_unit_{0};
    std::atomic<int> piece_limit_{0};             // pieces below it have a slot to go to
    std::atomic<bool> stop_{false};               // give up on the job (a HIP call failed)

    std::vector<std::thread> threads_;
    std::mutex m_;
    std::condition_variable wake_, idle_;
    int job_ = 0, busy_ = 0;
    bool quit_ = false;
};

}  // namespace cybq
