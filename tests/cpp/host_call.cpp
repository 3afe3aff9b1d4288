// HostCall (host_call.h) over a stand-in for the HIP runtime: live
// allocations are counted, freeing one that is not live fails the run, and a
// device reset frees everything, the next allocations taking the
// same addresses.  Run by tests/test_host_call.py.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "../../prrtc_amd/csrc/host_call.h"

namespace {
std::map<void *, unsigned long long> live;   // allocations, by number
unsigned long long last_id = 0;
int device = 0, fail_after = -1;   // allocations until one fails (-1: none)
alignas(256) char pool[64];

void check(bool ok, const char *what) {
    if (!ok) {
        std::printf("%s\n", what);
        std::exit(1);
    }
}
hipError_t take(void **p, int kind) {
    if (fail_after == 0) return hipErrorOutOfMemory;
    if (fail_after > 0) fail_after--;
    for (int i = kind; i < 64; i += 2)   // the lowest free address of the kind
        if (!live.count(pool + i)) {
            *p = pool + i;
            live[*p] = ++last_id;
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t give(void *p, const char *what) {
    check(live.erase(p) == 1, what);
    return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = device, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t) { return take(p, 0); }
hipError_t hipHostMalloc(void **p, size_t, unsigned) { return take(p, 1); }
hipError_t hipFree(void *p) { return give(p, "freed device memory that is not live"); }
hipError_t hipHostFree(void *p) { return give(p, "freed host memory that is not live"); }
hipError_t hipPointerGetAttribute(void *out, hipPointer_attribute a, hipDeviceptr_t p) {
    check(a == HIP_POINTER_ATTRIBUTE_BUFFER_ID, "attribute");
    if (!live.count(p)) return hipErrorInvalidValue;
    *static_cast<unsigned long long *>(out) = live[p];
    return hipSuccess;
}
}

static void usable(prrtc::HostCall &hc, size_t n) {
    check(hc.bytes >= n && live.count(hc.dev) && live.count(hc.host), "buffers are not live");
    check(live[hc.dev] == hc.dev_id && live[hc.host] == hc.host_id, "buffers are someone else's");
}

int main() {
    {
        prrtc::HostCall hc;
        hc.need(1000);
        usable(hc, 1000);
        const unsigned long long id = hc.dev_id;
        hc.need(2000);
        check(hc.dev_id == id && live.size() == 2, "a call that fits allocates nothing");
        hc.need(1 << 20);
        usable(hc, 1 << 20);
        check(live.size() == 2, "the old buffers are freed");
        device = 1;   // another device: buffers of its own
        hc.need(1000);
        usable(hc, 1000);
        check(hc.device == 1 && live.size() == 2, "one set is kept");

        live.clear();   // a device reset, and nothing since
        hc.need(1000);
        usable(hc, 1000);
        check(live.size() == 2, "a new set after a reset");
        live.clear();   // a reset, and another owner at the same addresses
        void *d, *h;
        check(!hipMalloc(&d, 8) && !hipHostMalloc(&h, 8, 0), "owner");
        check(d == hc.dev && h == hc.host, "the same addresses");
        hc.need(1000);
        usable(hc, 1000);
        check(live.size() == 4 && hc.dev != d && hc.host != h, "the owner keeps its own");
        hipFree(d), hipHostFree(h);

        for (int k = 0; k < 2; k++) {   // each allocation of a set fails: nothing is kept
            live.clear();
            fail_after = k;
            bool thrown = false;
            try {
                hc.need(1000);
            } catch (const prrtc::HipError &) {
                thrown = true;
            }
            fail_after = -1;
            check(thrown && live.empty() && hc.bytes == 0, "a failed set is given back");
        }
        hc.need(1000);
        usable(hc, 1000);
    }
    check(live.empty(), "everything is freed at the end");
    {
        prrtc::HostCall hc;
        hc.need(1000);
        live.clear();   // a reset before the thread ends
    }
    return 0;
}
