// pool.h - what tensors need besides their kernels, kept between tensors: device memory, and the pinned word + event
// through which a device-side scan reports back.
//
// hipMalloc + hipFree of a tensor cost 30 - 400 us and the free waits for the whole device; importing a small
// tensor takes a tenth of that.  One pool per device for the process (handles may outlive the context that made
// them), guarded by a mutex, bounded by kPoolBytes, emptied when the device's last context goes, when memory runs out or when the
// caller asks (cybq_trim).
//
// A block that comes back may still be read by work in flight.  `used_on` says where: kUnused, kDefaultStream (all of
// it went to the default stream), or kElsewhere.  It is handed out again without waiting only to a caller that
// writes it on the default stream and when all earlier use was there too - stream order does the rest; otherwise the
// device is synchronised first, which is what hipFree does.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace cybq {

enum UsedOn : int { kUnused = 0, kDefaultStream = 1, kElsewhere = 2 };

constexpr size_t kPoolBytes = (size_t)512 << 20;

hipError_t pool_retain(int device);     // a context lives on `device`
void pool_release(int device);          // ... and is gone

// `block` receives the size to hand back with the pointer.  `first_use`: where the caller writes it first.
hipError_t pool_alloc(int device, size_t bytes, UsedOn first_use, void** p, size_t* block);
void pool_free(int device, void* p, size_t block, UsedOn used_on);
hipError_t pool_trim(int device);       // everything kept goes back to the device

struct ScanSlot {
    uint32_t* word = nullptr;           // pinned host memory, device-visible
    hipEvent_t done = nullptr;
};
hipError_t scan_acquire(int device, ScanSlot* s);
void scan_release(int device, ScanSlot s);

}  // namespace cybq
