// host_stage.h -- copies of host images to the device through pinned memory.
//
// A two-dimensional copy from pageable memory goes through the runtime row by
// row: one 640x480 colour image took about 4.6 ms, and the frame loop made
// five such copies per frame (23 ms of a 23 ms frame).  Here the host copies
// the rows into one of two pinned slots and enqueues the slot's copy, so the
// caller's memory is free on return and one slot fills while the other is in
// flight.  The host waits only for a slot: an image of up to 2 MiB does not
// wait for the device unless the images before it are still on their way, but
// the third MiB of a larger one waits until the first has been copied, and so
// for the work queued ahead of it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>

#include "host_wait.h"

namespace slam {

class HostStage {
public:
    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    // The owner has synchronised the streams of its uploads.
    ~HostStage()
    {
        for (auto& s : slots_)
            if (s.ev) (void)hipEventDestroy(s.ev);
        if (pin_) (void)hipHostFree(pin_);
    }

    // The slots, with the owner's other memory, so that no upload allocates
    // (about 50 us): two of its largest image, at most 1 MiB each.
    hipError_t create(size_t largest)
    {
        slot_ = std::min(kSlot, (largest + 4095) / 4096 * 4096);
        if (hipError_t e = hipHostMalloc((void**)&pin_, 2 * slot_, hipHostMallocDefault)) {
            pin_ = nullptr;
            return e;
        }
        for (int k = 0; k < 2; ++k) {
            slots_[k].pin = pin_ + k * slot_;
            if (hipError_t e = hipEventCreateWithFlags(&slots_[k].ev, hipEventDisableTiming)) {
                slots_[k].ev = nullptr;
                return e;
            }
        }
        return hipSuccess;
    }

    // rows x row bytes at `src` (pitch bytes apart) to contiguous device
    // memory `dst`, in order on `s`.  Refused under stream capture, where a
    // replay would copy the slot's later contents.
    hipError_t upload(void* dst, const void* src, size_t pitch, size_t row, int rows, hipStream_t s)
    {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipError_t e = hipStreamIsCapturing(s, &cap)) return e;
        if (cap != hipStreamCaptureStatusNone) return hipErrorStreamCaptureUnsupported;
        const size_t total = row * (size_t)rows;
        for (size_t at = 0; at < total;) {
            Slot& q = slots_[next_];
            next_ ^= 1;
            if (hipError_t e = ready(q)) return e;
            const size_t n = std::min(slot_, total - at);
            for (size_t done = 0; done < n;) {
                const size_t y = (at + done) / row, x = (at + done) % row;
                const size_t m = pitch == row ? n - done : std::min(n - done, row - x);
                memcpy(q.pin + done, (const uint8_t*)src + y * pitch + x, m);
                done += m;
            }
            if (hipError_t e = hipMemcpyAsync((uint8_t*)dst + at, q.pin, n, hipMemcpyHostToDevice, s)) return e;
            if (hipError_t e = hipEventRecord(q.ev, s)) {
                (void)hipStreamSynchronize(s);   // the slot is free again, whatever became of the event
                return e;
            }
            q.used = true;
            at += n;
        }
        return hipSuccess;
    }

private:
    static constexpr size_t kSlot = (size_t)1 << 20;
    struct Slot {
        uint8_t* pin = nullptr;
        hipEvent_t ev = nullptr;
        bool used = false;
    };

    static hipError_t ready(Slot& q)
    {
        if (!q.used) return hipSuccess;
        if (hipError_t e = poll_event(q.ev)) return e;
        q.used = false;
        return hipSuccess;
    }

    uint8_t* pin_ = nullptr;
    size_t slot_ = 0;
    Slot slots_[2];
    int next_ = 0;
};

}  // namespace slam
