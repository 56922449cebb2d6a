// What streams of two devices wait for, against a HIP runtime that keeps a record instead of running anything.
#include "../deepep_efa_amd/csrc/event.hpp"

#include <cstdio>
#include <cstdlib>
#include <map>
#include <vector>

struct Event {
    unsigned flags = 0;
    hipStream_t recorded_on = nullptr;
    std::vector<Event*> behind;  // what that stream had waited for
    int device = -1;
    bool alive = true;
};
static int current_device = 0, next_stream = 100;
static std::map<hipStream_t, std::vector<Event*>> waits;  // by stream, in order
static std::map<hipStream_t, int> device_of;
static std::vector<Event*> events;

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = current_device, hipSuccess; }
hipError_t hipSetDevice(int d) { return current_device = d, hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "an error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(uintptr_t(next_stream++));
    return device_of[*s] = current_device, hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
    events.push_back(new Event{flags, nullptr, {}, current_device, true});
    return *e = reinterpret_cast<hipEvent_t>(events.back()), hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Event* event = reinterpret_cast<Event*>(e);
    if (device_of.at(s) != event->device) return hipErrorInvalidHandle;  // as HIP does
    return event->recorded_on = s, event->behind = waits[s], hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    return waits[s].push_back(reinterpret_cast<Event*>(e)), hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return reinterpret_cast<Event*>(e)->alive = false, hipSuccess; }
}

#define CHECK(cond) \
    if (!(cond)) return std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond), EXIT_FAILURE

int main() {
    const hipStream_t a = reinterpret_cast<hipStream_t>(uintptr_t(1)), b = reinterpret_cast<hipStream_t>(uintptr_t(2));
    const hipStream_t other = reinterpret_cast<hipStream_t>(uintptr_t(3));
    device_of[a] = device_of[b] = 0, device_of[other] = 1;
    using deep_ep::DeviceEvent;
    current_device = 1;
    for (int pass = 0; pass < 2; ++pass) {
        waits.clear();
        {
            const DeviceEvent local(0, a, DeviceEvent::kLocal);
            Event* const e = events.back();
            CHECK((e->flags & hipEventDisableSystemFence) != 0 && e->recorded_on == a && current_device == 1);
            local.wait_on(0, b);
            CHECK(waits[b] == std::vector<Event*>{e});
            local.wait_on(1, other);
            CHECK(waits[other].size() == 1 && waits[other][0] != e && current_device == 1);
            const Event& relayed = *waits[other][0];
            CHECK((relayed.flags & hipEventReleaseToSystem) != 0 && (relayed.flags & hipEventDisableSystemFence) == 0);
            CHECK(relayed.recorded_on != a && relayed.recorded_on != b);  // not behind what their callers gave them since
            CHECK(relayed.behind.size() == 1 && relayed.behind[0] == e);
        }
        waits.clear();
        {
            const DeviceEvent fenced(0, a, DeviceEvent::kSystem);
            Event* const e = events.back();
            CHECK((e->flags & hipEventDisableSystemFence) == 0);
            fenced.wait_on(1, other);
            CHECK(waits[other] == std::vector<Event*>{e});
        }
    }
    CHECK(next_stream == 101);  // one relay for the device
    for (const Event* e : events) CHECK(!e->alive);
    CHECK(current_device == 1);
    return EXIT_SUCCESS;
}
