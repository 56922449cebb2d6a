// Events that streams wait for (reference: csrc/event.hpp:9-25).  Streams are named by their device and HIP handle.
#pragma once
#include <c10/core/impl/GPUTrace.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <mutex>
#include <unordered_map>

#include "host_error.hpp"

namespace deep_ep {

// The calling thread's device, changed for a scope.
class ScopedDevice {
    int before = -1, during;

public:
    explicit ScopedDevice(int device) : during(device) {
        hip_check(hipGetDevice(&before), "event.hpp", __LINE__);
        if (before != during) hip_check(hipSetDevice(during), "event.hpp", __LINE__);
    }
    ScopedDevice(const ScopedDevice&) = delete;
    ~ScopedDevice() {
        if (before != during) (void)hipSetDevice(before);
    }
};

// An event that streams wait for, and nobody else: the handle cannot be queried, synchronised with or shared.  PyTorch's
// event callbacks (torch.cuda._gpu_trace) hear of it as of PyTorch's own.
// kLocal: recorded without the system-scope fence (hipEventDisableSystemFence), which writes the caches back and invalidates
// them between two kernels and without which memory may not be visible to the host and other devices.  Streams of the
// device need none, they see one another's writes when the kernels that made them have ended, and a host that reads behind
// one of them has the fence of its wait or copy.  A stream of another device waits for a second event instead, which a
// stream of this one records behind the first, with the fence.
class DeviceEvent {
public:
    enum Scope : unsigned { kSystem = 0, kLocal = hipEventDisableSystemFence, kSystemAlways = hipEventReleaseToSystem };

private:
    hipEvent_t event = nullptr;
    const int device;
    const Scope scope;

    template <typename F>
    static void trace(F report) {
        if (const auto* interpreter = c10::impl::GPUTrace::get_trace()) report(**interpreter);
    }
    uintptr_t name() const { return reinterpret_cast<uintptr_t>(event); }
    void destroy() {
        trace([&](const auto& to) { to.trace_gpu_event_deletion(c10::kCUDA, name()); });
        (void)hipEventDestroy(event);
    }

    // The one stream of the current device on which events are recorded for other devices; kept until the process ends.
    // What several threads put there at once may wait for one another's events, never for anything that follows them.
    static hipStream_t relay_of(int device) {
        static std::mutex& mutex = *new std::mutex;
        static auto& streams = *new std::unordered_map<int, hipStream_t>;
        const std::lock_guard<std::mutex> lock(mutex);  // not held beyond: the callbacks below run Python
        hipStream_t& relay = streams[device];
        if (relay == nullptr) hip_check(hipStreamCreateWithFlags(&relay, hipStreamNonBlocking), "event.hpp", __LINE__);
        return relay;
    }

    void stream_waits(hipStream_t waiter) const {
        trace([&](const auto& to) {
            to.trace_gpu_event_wait(c10::kCUDA, name(), reinterpret_cast<uintptr_t>(waiter));
        });
        hip_check(hipStreamWaitEvent(waiter, event, 0), "event.hpp", __LINE__);
    }

public:
    DeviceEvent(int device, hipStream_t stream, Scope scope) : device(device), scope(scope) {
        const ScopedDevice current(device);
        hip_check(hipEventCreateWithFlags(&event, hipEventDisableTiming | scope), "event.hpp", __LINE__);
        try {
            trace([&](const auto& to) {
                to.trace_gpu_event_creation(c10::kCUDA, name());
                to.trace_gpu_event_record(c10::kCUDA, name(), reinterpret_cast<uintptr_t>(stream));
            });
            hip_check(hipEventRecord(event, stream), "event.hpp", __LINE__);
        } catch (...) {
            destroy();
            throw;
        }
    }
    DeviceEvent(const DeviceEvent&) = delete;
    ~DeviceEvent() {
        try {
            const ScopedDevice current(device);
            destroy();
        } catch (...) {  // the process is ending
        }
    }

    void wait_on(int waiter_device, hipStream_t waiter) const {
        if (scope == kLocal && waiter_device != device) {
            const ScopedDevice current(device);
            const hipStream_t relay = relay_of(device);
            stream_waits(relay);
            DeviceEvent(device, relay, kSystemAlways).wait_on(waiter_device, waiter);
            return;
        }
        const ScopedDevice current(waiter_device);
        stream_waits(waiter);
    }
};

}  // namespace deep_ep
