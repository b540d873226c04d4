// lulesh_transfer.hpp -- fields between host memory and the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <mutex>

namespace lulesh {

// one field of a transfer; host memory holds float64 values
struct TransferItem {
    void *dev;
    double *host;           // only read on the way to the device
    int64_t n;
    bool f32;               // the device holds float32
    const int32_t *place;   // device list: place of each value in the field, or null
};

// Moves lists of fields through a ring of pinned staging slots: while the
// copy engine fills or drains one slot, threads move others to or from the
// caller's memory.  A copy straight to pageable memory runs on one thread,
// which also takes the page faults of a buffer just allocated.
//
// One per domain; the slots are made at its first transfer, of the size of its
// largest field and at most kSlotBytes.  Calls are serialised.  run() returns
// after the last value is in place; `stream` orders the transfer after work
// queued earlier.
class FieldTransfer {
public:
    static constexpr size_t kSlotBytes = size_t(4) << 20;
    static constexpr int kSlots = 8;

    ~FieldTransfer();
    hipError_t run(const TransferItem *items, int count, bool to_device, hipStream_t stream);

private:
    hipError_t reserve(size_t bytes, bool placed);
    hipError_t move_all(const TransferItem *items, int count, bool to_device,
                        hipStream_t stream);

    std::mutex lock_;
    char *slots_ = nullptr;
    size_t slot_bytes_ = 0;
    bool pinned_ = false;
    char *dev_slots_ = nullptr;  // the values of a renumbered field, in the caller's order
    hipEvent_t events_[kSlots] = {};
};

}  // namespace lulesh
