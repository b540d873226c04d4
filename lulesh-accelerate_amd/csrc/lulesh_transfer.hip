// lulesh_transfer.hip -- see lulesh_transfer.hpp.
//
// The state of a 150^3 domain (11 fields, 300 MB) to newly allocated arrays
// and back: 7.2 and 6.9 ms, the rate of the copy engine over the bus (44
// GB/s); one pageable copy after another took 33 and 10.4 ms.  240^3 28.5 and
// 26.5 ms (119, 42), 60^3 1.1 and 0.7 (4.5, 1.0), 10^3 0.16 and 0.17 (0.32,
// 0.26).  Slots of 2 MB: 150^3 8.4 and 7.7 ms.
#include "lulesh_transfer.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace lulesh {

namespace {

// Below this one thread does it: starting the others costs more.  A single
// field below it needs no slots either: 27000 values straight to a new array
// take 78 us, through a slot 94; the 48 fields of eight members of 60^3 to
// 90^3 14.3 and 17.3 ms.
constexpr size_t kThreadedBytes = size_t(4) << 20;
constexpr int kThreads = 8;

// The fields of a state of middling size go straight to and from the caller's
// memory as well: below kDirectField a copy to pageable memory has a fixed cost
// above a slot's, and from kDirectBytes on the threads win.  Through slots and
// straight, in ms: uploads 10^3 0.165 and 0.17, 14^3 0.245 and 0.225, 30^3 0.29
// and 0.23, 45^3 0.51 and 0.355, 50^3 0.545 and 0.48, 60^3 0.72 and 0.72; a
// domain's first download, which makes the slots, 10^3 0.18 and 0.22, 14^3 0.27
// and 0.155, 30^3 0.33 and 0.27, 45^3 0.82 and 0.62; later ones 50^3 0.67 and
// 0.9, 60^3 0.8 and 1.2.
constexpr size_t kDirectField = size_t(16) << 10;
constexpr size_t kDirectBytes = size_t(10) << 20;

__global__ __launch_bounds__(256) void k_gather(const double *field, const int32_t *place,
                                                double *out, int n)
{
    const int i = int(blockIdx.x) * 256 + int(threadIdx.x);
    if (i < n) {
        out[i] = field[place[i]];
    }
}

__global__ __launch_bounds__(256) void k_scatter(double *field, const int32_t *place,
                                                 const double *in, int n)
{
    const int i = int(blockIdx.x) * 256 + int(threadIdx.x);
    if (i < n) {
        field[place[i]] = in[i];
    }
}

// the values [first, first + n) of an item
struct Chunk {
    const TransferItem *item;
    int64_t first;
    int n;
};

size_t device_bytes(const TransferItem &t) { return t.f32 ? sizeof(float) : sizeof(double); }

// caller's memory -> slot
void fill_slot(const Chunk &c, char *slot)
{
    const double *src = c.item->host + c.first;
    if (!c.item->f32) {
        std::memcpy(slot, src, size_t(c.n) * sizeof(double));
        return;
    }
    float *dst = reinterpret_cast<float *>(slot);
    for (int i = 0; i < c.n; ++i) {
        dst[i] = static_cast<float>(src[i]);
    }
}

// slot -> caller's memory
void drain_slot(const Chunk &c, const char *slot)
{
    double *dst = c.item->host + c.first;
    if (!c.item->f32) {
        std::memcpy(dst, slot, size_t(c.n) * sizeof(double));
        return;
    }
    const float *src = reinterpret_cast<const float *>(slot);
    for (int i = 0; i < c.n; ++i) {
        dst[i] = static_cast<double>(src[i]);
    }
}

}  // namespace

FieldTransfer::~FieldTransfer()
{
    for (hipEvent_t e : events_) {
        if (e) (void)hipEventDestroy(e);
    }
    if (slots_ && pinned_) (void)hipHostFree(slots_);
    if (slots_ && !pinned_) std::free(slots_);
    if (dev_slots_) (void)hipFree(dev_slots_);
}

// slots that hold a field of `bytes`, kSlotBytes at most; between transfers,
// so nothing uses the old ones
hipError_t FieldTransfer::reserve(size_t bytes, bool placed)
{
    for (hipEvent_t &e : events_) {
        if (!e) {
            const hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
            if (r != hipSuccess) return r;
        }
    }
    const size_t want = std::min(kSlotBytes, (bytes + 4095) / 4096 * 4096);
    if (!slots_ || slot_bytes_ < want) {
        if (slots_ && pinned_) (void)hipHostFree(slots_);
        if (slots_ && !pinned_) std::free(slots_);
        slots_ = nullptr;
        if (dev_slots_) (void)hipFree(dev_slots_);
        dev_slots_ = nullptr;
        void *p = nullptr;
        pinned_ = hipHostMalloc(&p, kSlots * want, hipHostMallocDefault) == hipSuccess;
        if (!pinned_) {
            // copies through ordinary memory are slower, and as correct
            (void)hipGetLastError();
            p = std::malloc(kSlots * want);
            if (!p) return hipErrorOutOfMemory;
        }
        slots_ = static_cast<char *>(p);
        slot_bytes_ = want;
    }
    if (placed && !dev_slots_) {
        void *p = nullptr;
        const hipError_t r = hipMalloc(&p, kSlots * slot_bytes_);
        if (r != hipSuccess) return r;
        dev_slots_ = static_cast<char *>(p);
    }
    return hipSuccess;
}

hipError_t FieldTransfer::run(const TransferItem *items, int count, bool to_device,
                              hipStream_t stream)
{
    const std::lock_guard<std::mutex> guard(lock_);
    // fields that share host memory are written one after another
    bool shared = false;
    for (int i = 0; i < count && !to_device; ++i) {
        for (int j = 0; j < i; ++j) {
            shared = shared || (items[i].host < items[j].host + items[j].n &&
                                items[j].host < items[i].host + items[i].n);
        }
    }
    if (!shared) {
        return move_all(items, count, to_device, stream);
    }
    hipError_t err = hipSuccess;
    for (int i = 0; i < count && err == hipSuccess; ++i) {
        err = move_all(items + i, 1, to_device, stream);
    }
    return err;
}

hipError_t FieldTransfer::move_all(const TransferItem *items, int count, bool to_device,
                                   hipStream_t stream)
{
    size_t bytes = 0, largest = 0;
    bool placed = false, plain = true;
    for (int i = 0; i < count; ++i) {
        plain = plain && !items[i].f32 && !items[i].place;
        const size_t b = size_t(items[i].n) * device_bytes(items[i]);
        bytes += b;
        largest = std::max(largest, b);
        placed = placed || items[i].place;
    }
    if (bytes == 0) {
        return hipStreamSynchronize(stream);
    }
    const bool direct = plain && (count == 1 ? bytes < kThreadedBytes
                                             : largest >= kDirectField && bytes < kDirectBytes);
    if (direct) {
        hipError_t r = hipSuccess;
        for (int i = 0; i < count && r == hipSuccess; ++i) {
            void *const host = items[i].host;
            const size_t b = size_t(items[i].n) * sizeof(double);
            r = to_device ? hipMemcpyAsync(items[i].dev, host, b, hipMemcpyHostToDevice, stream)
                          : hipMemcpyAsync(host, items[i].dev, b, hipMemcpyDeviceToHost, stream);
            // one by one: 18^3 0.16 ms, all queued before one wait 0.195
            if (r == hipSuccess && !to_device) r = hipStreamSynchronize(stream);
        }
        const hipError_t end = hipStreamSynchronize(stream);
        return r != hipSuccess ? r : end;
    }
    hipError_t err = reserve(largest, placed);
    if (err != hipSuccess) {
        return err;
    }
    std::vector<Chunk> chunks;
    try {
        for (int i = 0; i < count; ++i) {
            const int64_t most = int64_t(slot_bytes_ / device_bytes(items[i]));
            for (int64_t f = 0; f < items[i].n; f += most) {
                chunks.push_back({&items[i], f, int(std::min(most, items[i].n - f))});
            }
        }
    } catch (const std::bad_alloc &) {
        return hipErrorOutOfMemory;
    }
    const int total = int(chunks.size());
    auto slot = [&](int c) { return slots_ + size_t(c % kSlots) * slot_bytes_; };
    // the copy between slot and field, and the event after it
    auto issue = [&](int c) -> hipError_t {
        const Chunk &k = chunks[size_t(c)];
        const TransferItem &t = *k.item;
        const size_t b = size_t(k.n) * device_bytes(t);
        char *field = static_cast<char *>(t.dev) + size_t(k.first) * device_bytes(t);
        double *stage = nullptr;
        if (t.place) {
            stage = reinterpret_cast<double *>(dev_slots_ + size_t(c % kSlots) * slot_bytes_);
        }
        const unsigned grid = unsigned((k.n + 255) / 256);
        hipError_t r = hipSuccess;
        if (to_device) {
            r = hipMemcpyAsync(stage ? static_cast<void *>(stage) : field, slot(c), b,
                               hipMemcpyHostToDevice, stream);
            if (r == hipSuccess && stage) {
                hipLaunchKernelGGL(k_scatter, dim3(grid), dim3(256), 0, stream,
                                   static_cast<double *>(t.dev), t.place + k.first, stage, k.n);
                r = hipGetLastError();
            }
        } else {
            if (stage) {
                hipLaunchKernelGGL(k_gather, dim3(grid), dim3(256), 0, stream,
                                   static_cast<const double *>(t.dev), t.place + k.first, stage,
                                   k.n);
                r = hipGetLastError();
            }
            if (r == hipSuccess) {
                r = hipMemcpyAsync(slot(c), stage ? static_cast<void *>(stage) : field, b,
                                   hipMemcpyDeviceToHost, stream);
            }
        }
        return r != hipSuccess ? r : hipEventRecord(events_[c % kSlots], stream);
    };

    // This thread issues the chunks in order; the others move them between
    // slots and the caller's memory.  `issued` and `moved[]` are guarded by m.
    std::mutex m;
    std::condition_variable cv;
    int issued = 0;
    std::vector<char> moved;
    std::vector<std::thread> threads;
    std::atomic<int> next{0};
    bool failed = false;
    // The host's part of chunk c.  To the device: wait for the copy that
    // read the slot last, then fill it.  From it: wait for the copy, then
    // drain the slot.
    auto move = [&](int c) -> hipError_t {
        const bool wait = !to_device || c >= kSlots;
        const hipError_t r = wait ? hipEventSynchronize(events_[c % kSlots]) : hipSuccess;
        if (r == hipSuccess) {
            to_device ? fill_slot(chunks[size_t(c)], slot(c))
                      : drain_slot(chunks[size_t(c)], slot(c));
        }
        return r;
    };
    auto work = [&] {
        for (;;) {
            const int c = next.fetch_add(1);
            if (c >= total) return;
            {
                std::unique_lock<std::mutex> l(m);
                cv.wait(l, [&] { return failed || issued > (to_device ? c - kSlots : c); });
                if (failed) return;
            }
            const hipError_t r = move(c);
            const std::lock_guard<std::mutex> l(m);
            moved[size_t(c)] = 1;
            if (r != hipSuccess) {
                failed = true;
                err = r;
            }
            cv.notify_all();
        }
    };
    if (bytes >= kThreadedBytes && total > 1) {
        const int most = std::min({kThreads, total, int(std::thread::hardware_concurrency())});
        try {
            moved.assign(size_t(total), 0);
            threads.reserve(size_t(std::max(most, 0)));
            for (int i = 0; i < most; ++i) {
                threads.emplace_back(work);
            }
        } catch (const std::exception &) {
            // with as many as there are
        }
    }
    if (threads.empty()) {
        for (int c = 0; c < total + kSlots && err == hipSuccess; ++c) {
            if (to_device) {
                if (c < total && (err = move(c)) == hipSuccess) err = issue(c);
            } else {
                if (c >= kSlots) err = move(c - kSlots);
                if (c < total && err == hipSuccess) err = issue(c);
            }
        }
    } else {
        for (int c = 0; c < total; ++c) {
            {
                // to the device: the slot is filled; from it: it is drained
                const int before = to_device ? c : c - kSlots;
                std::unique_lock<std::mutex> l(m);
                cv.wait(l, [&] { return failed || before < 0 || moved[size_t(before)]; });
                if (failed) break;
            }
            const hipError_t r = issue(c);
            const std::lock_guard<std::mutex> l(m);
            ++issued;
            if (r != hipSuccess) {
                failed = true;
                err = r;
            }
            cv.notify_all();
        }
        for (std::thread &t : threads) {
            t.join();
        }
    }
    const hipError_t end = hipStreamSynchronize(stream);
    return err != hipSuccess ? err : end;
}

}  // namespace lulesh
