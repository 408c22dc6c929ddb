// What lq_encode_chunks reads back: two words of pinned host memory that the
// launches write, and an event after the launch that writes the last one.
// Slots are taken for one call and given back at its end, to the device they
// belong to; up to kReadSlots wait for the next call, the others are freed.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <thread>

namespace lq {

struct ReadSlot {
    int64_t* host = nullptr;
    hipEvent_t event = nullptr;
    int device = -1;
};

constexpr int kReadSlots = 16;

struct ReadPool {
    std::atomic_flag busy = ATOMIC_FLAG_INIT;   // held for a scan of the slots
    ReadSlot slots[kReadSlots];                 // host null: free place

    void lock() { while (busy.test_and_set(std::memory_order_acquire)) std::this_thread::yield(); }
    void unlock() { busy.clear(std::memory_order_release); }

    // A slot whose event can be recorded on stream s: an event belongs to the
    // device that is current when it is made, which need not be the stream's.
    bool take(hipStream_t s, ReadSlot* out) {
        hipDevice_t dev = 0;
        if (hipStreamGetDevice(s, &dev) != hipSuccess) return false;
        ReadSlot r;
        lock();
        for (ReadSlot& p : slots)
            if (p.host && p.device == dev) {
                r = p;
                p = ReadSlot();
                break;
            }
        unlock();
        if (!r.host && !make(dev, &r)) return false;
        *out = r;
        return true;
    }
    void give(const ReadSlot& r) {
        lock();
        for (ReadSlot& p : slots)
            if (!p.host) {
                p = r;
                unlock();
                return;
            }
        unlock();
        (void)hipEventDestroy(r.event);
        (void)hipHostFree(r.host);
    }

  private:
    static bool make(int dev, ReadSlot* r) {
        int current = 0;
        if (hipGetDevice(&current) != hipSuccess) return false;
        if (current != dev && hipSetDevice(dev) != hipSuccess) return false;
        r->device = dev;
        bool ok = hipHostMalloc(reinterpret_cast<void**>(&r->host), 2 * sizeof(int64_t), hipHostMallocDefault) == hipSuccess;
        if (ok && hipEventCreateWithFlags(&r->event, hipEventDisableTiming) != hipSuccess) {
            (void)hipHostFree(r->host);
            ok = false;
        }
        if (current != dev) (void)hipSetDevice(current);
        return ok;
    }
};

}  // namespace lq
