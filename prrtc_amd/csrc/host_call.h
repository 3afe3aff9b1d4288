// What a thread's verdict calls on host buffers keep between calls.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>

namespace prrtc {

struct HipError {
    hipError_t code;
    const char *where;
};

#define PRRTC_HIP(call)                                                   \
    do {                                                                  \
        hipError_t _e = (call);                                           \
        if (_e != hipSuccess) throw ::prrtc::HipError{_e, #call};         \
    } while (0)

// Device buffer and pinned staging of a thread's host-buffer calls
// (check_poses, validate_edges), kept between calls: three device
// allocations and frees and three blocking copies were 110 of the 150 us of
// a 4096-pose check.  At most kMost bytes of each, released when the thread
// ends; a larger call brings its own (verdict_call).  Every call waits for
// its own work, so a buffer is never in use when the thread's next call takes
// it.  The calls run on the null stream: a process has four hardware queues,
// and a stream kept here took one of them, so that two robot classes of a
// server shared another and their slices ran one after the other (500
// requests/s, median latency 3.6 -> 4.4 ms).
//
// A program may reset the device between two calls, which frees both buffers;
// their addresses may then be anyone's.  The runtime gives every allocation a
// number of its own for the life of the process, so the buffers are asked for
// theirs (0.07 us each) before they are used or freed, and are forgotten if it
// is another's.
struct HostCall {
    static constexpr size_t kMost = 16u << 20;
    char *dev = nullptr, *host = nullptr;
    size_t bytes = 0;   // of each
    int device = -1;   // of the buffers
    unsigned long long dev_id = 0, host_id = 0;

    // Number of the allocation that holds p; 0: none.
    static unsigned long long buffer_id(void *p) {
        unsigned long long id = 0;
        if (p && hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, (hipDeviceptr_t)p) == hipSuccess) return id;
        (void)hipGetLastError();   // not for the next call's check to find
        return 0;
    }
    bool intact() const { return dev && buffer_id(dev) == dev_id && buffer_id(host) == host_id; }
    void release() {
        if (intact()) {
            (void)hipHostFree(host);
            (void)hipFree(dev);
        }
        dev = host = nullptr;
        bytes = 0;
        device = -1;
    }
    // Both buffers of at least n <= kMost bytes on the thread's current device.
    void need(size_t n) {
        int cur = 0;
        PRRTC_HIP(hipGetDevice(&cur));
        if (cur == device && n <= bytes && intact()) return;
        release();
        const size_t size = std::min(kMost, n + n / 2 + 65536);
        char *d = nullptr, *h = nullptr;
        PRRTC_HIP(hipMalloc(reinterpret_cast<void **>(&d), size));
        try {
            PRRTC_HIP(hipHostMalloc(reinterpret_cast<void **>(&h), size, hipHostMallocDefault));
        } catch (...) {   // both or none are kept
            (void)hipFree(d);
            throw;
        }
        dev = d;
        host = h;
        bytes = size;
        device = cur;
        dev_id = buffer_id(dev);
        host_id = buffer_id(host);
    }

    HostCall() = default;
    ~HostCall() { release(); }
    HostCall(const HostCall &) = delete;
    HostCall &operator=(const HostCall &) = delete;
};

}  // namespace prrtc
